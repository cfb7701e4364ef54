"""The transforms whose speed is measured: spin spherical-harmonic and Wigner
transforms on one GPU, through the public entry points of ``s2fft_amd``.

``listed()`` are the cases, ``draw(rng)`` gives more of the same ranges,
``prepare`` / ``run`` set one up and run one pass of it, ``work`` says what a
pass cannot do without and ``exact`` what it returns in 64-bit arithmetic.
Inputs and exact values come from a plain torch synthesis in this file
(Wigner-d recursion over l, dense azimuthal sums), not from the library.

What a case is (``kind``):

* ``forward`` / ``inverse``: ``s2fft_amd.forward`` / ``inverse`` on device
  tensors, ``batch`` maps per call; HEALPix forwards with ``iter`` steps of
  refinement.  ``precision`` other than "fp64": the same inverse on the
  matrix-core kernels of that precision.
* ``refine``: the mixed-precision conjugate-gradient forward of band-limited
  HEALPix maps with the learned preconditioner.
* ``forward_gradient``: d/df of sum |forward(f) - t|^2 (Gauss-Legendre);
  ``inverse_gradient``: d/dflm of sum |inverse(flm) - t|^2.
* ``wigner_forward`` / ``wigner_inverse`` / ``wigner_gradient``: the SO(3)
  transforms and d/dflmn of sum |inverse(flmn) - t|^2.
* ``precompute_forward``: the forward with a stored kernel that the caller keeps.
"""

import math

import numpy as np
import torch

import s2fft_amd
from s2fft_amd.learned.precond import MLPPreconditioner
from s2fft_amd.transforms import refine
from s2fft_amd.transforms import spherical as sph

DEVICE = "cuda:0"


def _case(kind, sampling, L, batch=1, spin=0, reality=False, nside=0, iter=0, N=0,
          precision="fp64"):
    return {"kind": kind, "sampling": sampling, "L": L, "batch": batch, "spin": spin,
            "reality": reality, "nside": nside, "iter": iter, "N": N, "precision": precision}


def listed():
    named = [
        # one small map inside an optimisation or sampling loop: launches and latency
        ("mw_inverse_L64", _case("inverse", "mw", 64)),
        # the analysis of one map at a common working resolution
        ("mw_forward_L128", _case("forward", "mw", 128)),
        # a batch of spin-2 (polarisation, shear) simulations, both directions;
        # the inverse in the reduced precision that such batches may choose
        ("mw_forward_L512_s2_b64", _case("forward", "mw", 512, 64, 2)),
        ("mw_inverse_L512_s2_b64_bf16", _case("inverse", "mw", 512, 64, 2, precision="bf16")),
        # odd band-limit, few maps, the symmetric equiangular grid
        ("mwss_forward_L193_s1_b3", _case("forward", "mwss", 193, 3, 1)),
        # one large sky map analysed with the usual three refinement steps
        ("hp_forward_n512_iter3", _case("forward", "healpix", 1024, reality=True, nside=512,
                                        iter=3)),
        # a handful of maps, nside not a power of two, odd band-limit above 2 nside
        ("hp_forward_n192_L449_b5_iter3", _case("forward", "healpix", 449, 5, reality=True,
                                                nside=192, iter=3)),
        # polarisation simulations on the sky pixelisation
        ("hp_inverse_n256_s2_b4", _case("inverse", "healpix", 512, 4, 2, nside=256)),
        # the largest: a batch of full-resolution maps to 1e-7, mixed precision
        ("hp_refine_n1024_b16", _case("refine", "healpix", 2048, 16, reality=True, nside=1024)),
        # the transforms inside a differentiable model: analysis and SO(3) synthesis
        ("gl_forward_gradient_L256", _case("forward_gradient", "gl", 256)),
        ("wigner_gradient_L64_N4", _case("wigner_gradient", "mw", 64, N=4)),
        # many maps of one band-limit with a kernel computed once
        ("hp_precompute_n64_b16", _case("precompute_forward", "healpix", 128, 16, reality=True,
                                        nside=64)),
    ]
    return [dict(c, name=name) for name, c in named]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("forward", "forward", "inverse", "inverse", "healpix_forward",
                       "healpix_forward", "healpix_inverse", "refine", "forward_gradient",
                       "inverse_gradient", "wigner", "precompute_forward"))
    spin = rng.choice((0, 0, 1, 2, -2))
    reality = spin == 0 and rng.random() < 0.5
    if kind in ("forward", "inverse"):
        sampling = rng.choice(("mw", "mw", "mwss", "dh", "gl"))
        L = _log_int(rng, 24, 700)
        batch = _log_int(rng, 1, max(1, min(64, 16 * (512 / L) ** 3)))
        precision = rng.choice(("fp64", "fp64", "bf16")) if kind == "inverse" else "fp64"
        return _case(kind, sampling, L, batch, spin, reality, precision=precision)
    if kind in ("healpix_forward", "healpix_inverse"):
        nside = _log_int(rng, 16, 512)
        L = int(nside * rng.uniform(2.0, 2.9))
        batch = _log_int(rng, 1, max(1, min(16, 4 * (512 / L) ** 3)))
        if kind == "healpix_inverse":
            return _case("inverse", "healpix", L, batch, spin, reality, nside)
        return _case("forward", "healpix", L, batch, spin, reality, nside,
                     iter=rng.choice((0, 1, 3)))
    if kind == "refine":
        nside = _log_int(rng, 128, 700)
        return _case("refine", "healpix", 2 * nside, rng.randint(4, 16), reality=True,
                     nside=nside)
    if kind == "forward_gradient":
        return _case(kind, "gl", _log_int(rng, 32, 400), rng.randint(1, 4), spin, reality)
    if kind == "inverse_gradient":
        if rng.random() < 0.5:
            nside = _log_int(rng, 16, 160)
            return _case(kind, "healpix", 2 * nside, rng.randint(1, 4), spin, reality, nside)
        return _case(kind, rng.choice(("mw", "mwss", "gl")), _log_int(rng, 32, 400),
                     rng.randint(1, 4), spin, reality)
    if kind == "wigner":
        return _case("wigner_" + rng.choice(("forward", "inverse", "gradient")),
                     rng.choice(("mw", "mwss")), _log_int(rng, 16, 128), N=rng.randint(2, 6))
    nside = _log_int(rng, 8, 64)
    return _case(kind, "healpix", 2 * nside, rng.randint(1, 16), spin, reality, nside)


# ------------------------------------------------------------ plain synthesis
def _grid(sampling, L, nside):
    """Colatitudes of the rings, and groups (rows, n, h, first pixels) of rings
    with n pixels at phi_p = pi (2 p + h) / n."""
    t = np.arange
    if sampling == "healpix":
        theta, n, h = [], [], []
        for r in range(1, 4 * nside):
            i = min(r, 4 * nside - r)
            if i < nside:
                z = 1.0 - i * i / (3.0 * nside * nside)
                theta.append(math.acos(z if r < 2 * nside else -z))
                n.append(4 * i)
                h.append(1)
            else:
                theta.append(math.acos(4.0 / 3.0 - 2.0 * r / (3.0 * nside)))
                n.append(4 * nside)
                h.append((r - nside + 1) % 2)
        theta, n, h = np.array(theta), np.array(n), np.array(h)
    else:
        theta = {"mw": lambda: (2 * t(L) + 1) * np.pi / (2 * L - 1),
                 "mwss": lambda: t(L + 1) * np.pi / L,
                 "dh": lambda: (2 * t(2 * L) + 1) * np.pi / (4 * L),
                 "gl": lambda: np.arccos(np.polynomial.legendre.leggauss(L)[0])[::-1]}[sampling]()
        n = np.full(len(theta), 2 * L if sampling == "mwss" else 2 * L - 1)
        h = np.zeros(len(theta), dtype=int)
    first = np.cumsum(n) - n
    groups = {}
    for r in range(len(theta)):
        groups.setdefault((int(n[r]), int(h[r])), []).append(r)
    return theta, [(rows, k[0], k[1], first[rows]) for k, rows in groups.items()], int(n.sum())


def _orders(L, reality):
    """The m of the columns below: by |m|, so that the active ones lead."""
    return list(range(L)) if reality else [0] + [s * m for m in range(1, L) for s in (1, -1)]


def _wigner_d(L, ms, n, theta, block=32):
    """Blocks (l, d) of d^l_{m, n}(theta), d[l - l_block, m, t], l ascending."""
    m = torch.tensor(ms, dtype=torch.float64, device=DEVICE)
    th = torch.tensor(np.ascontiguousarray(theta), device=DEVICE)
    x = torch.cos(th)
    lc, ls = torch.log(torch.cos(th / 2).abs()), torch.log(torch.sin(th / 2).abs())
    # logarithms of factorials in extended precision
    lf = np.concatenate([[0], np.cumsum(np.log(np.arange(1, 2 * L + 1, dtype=np.longdouble)))])
    start, scale = [], 460.0  # d is held times e^460 against underflow
    for q in ms:
        j, an = max(abs(q), abs(n)), abs(n)
        k, ecos, sgn = n, j + n, (-1) ** (j - n)
        if abs(q) >= an and q < 0:
            ecos, sgn = j - n, 1
        elif abs(q) < an:
            k, ecos, sgn = (q, j + q, 1) if n > 0 else (q, j - q, (-1) ** (j + q))
        start.append((float((lf[2 * j] - lf[j + abs(k)] - lf[j - abs(k)]) / 2), ecos, 2 * j - ecos,
                      sgn))
    st = torch.tensor(start, dtype=torch.float64, device=DEVICE)

    def power(e, logs):
        return torch.where(e == 0, torch.zeros_like(logs), e * logs)

    d = torch.zeros((len(ms), len(theta)), dtype=torch.float64, device=DEVICE)
    prev = torch.zeros_like(d)
    seen = 0
    for l0 in range(0, L, block):
        out = torch.zeros((min(block, L - l0),) + tuple(d.shape), dtype=torch.float64,
                          device=DEVICE)
        for l in range(l0, min(l0 + block, L)):
            if l < abs(n):
                continue
            now = min(len(ms), (l + 1) if len(ms) == L else 2 * l + 1)
            if now > seen:
                s = st[seen:now]
                d[seen:now] = s[:, 3:] * torch.exp(
                    s[:, :1] + power(s[:, 1:2], lc[None]) + power(s[:, 2:3], ls[None]) + scale)
                seen = now
            out[l - l0, :now] = d[:now]
            mm = m[:now]
            root = torch.sqrt(((l + 1.0) ** 2 - mm * mm) * ((l + 1.0) ** 2 - n * n))
            a = (2 * l + 1.0) * (l + 1.0) / root
            if l > 0:
                b = (2 * l + 1.0) * mm * n / (l * root)
                c = (l + 1.0) * torch.sqrt((l * l - mm * mm) * (l * l - n * n)) / (l * root)
            else:
                b, c = torch.zeros_like(a), torch.zeros_like(a)
            nxt = torch.addcmul(-c[:, None] * prev[:now], a[:, None] * x - b[:, None], d[:now])
            prev[:now] = d[:now]
            d[:now] = nxt
        yield l0, out.mul_(math.exp(-scale))


def _phases(ms, n, h):
    """e^{i m phi_p} of a ring, [m, p], from exactly reduced angles."""
    k = torch.tensor(ms, device=DEVICE)[:, None] * (2 * torch.arange(n, device=DEVICE) + h)
    ang = (k % (2 * n)).to(torch.float64) * (math.pi / n)
    return torch.polar(torch.ones_like(ang), ang)


def _norm(L):
    return torch.sqrt((2 * torch.arange(L, device=DEVICE, dtype=torch.float64) + 1) / (4 * math.pi))


def _synthesis(flm, spin, sampling, nside, reality, norm=None, ring_weight=None):
    """sum flm sY_lm on the pixels: (B, L, 2L-1) -> (B, npix)."""
    B, L = flm.shape[:2]
    theta, groups, npix = _grid(sampling, L, nside)
    ms = _orders(L, reality)
    x = flm[:, :, torch.tensor(ms, device=DEVICE) + L - 1] * (
        (-1) ** spin * (_norm(L) if norm is None else norm))[None, :, None]
    x = torch.view_as_real(x.permute(2, 1, 0).contiguous()).reshape(len(ms), L, 2 * B)
    F = torch.zeros((len(ms), len(theta), 2 * B), dtype=torch.float64, device=DEVICE)
    for l0, d in _wigner_d(L, ms, -spin, theta):
        F.baddbmm_(d.permute(1, 2, 0), x[:, l0:l0 + d.shape[0]].contiguous())
    if ring_weight is not None:
        F *= ring_weight[None, :, None]
    F = torch.view_as_complex(F.reshape(len(ms), len(theta), B, 2)).permute(2, 1, 0)
    f = torch.zeros((B, npix), dtype=torch.float64 if reality else torch.complex128,
                    device=DEVICE)
    if reality:
        F = torch.cat([F[..., :1], 2 * F[..., 1:]], -1)
    for rows, n, h, first in groups:
        E = _phases(ms, n, h)
        at = torch.from_numpy(first[:, None] + np.arange(n)).to(DEVICE)
        G = F[:, rows].reshape(-1, len(ms))
        v = G.real @ E.real - G.imag @ E.imag if reality else G @ E
        f[:, at.reshape(-1)] = v.reshape(B, -1)
    return f


def _projection(f, L, spin, sampling, nside, reality, weight, norm=None):
    """The conjugate transpose of _synthesis with a weight per ring: (B, npix)
    -> (B, L, 2L-1); real maps: m >= 0 and its conjugate half."""
    B = f.shape[0]
    theta, groups, _ = _grid(sampling, L, nside)
    ms = _orders(L, reality)
    F = torch.zeros((B, len(theta), len(ms)), dtype=torch.complex128, device=DEVICE)
    for rows, n, h, first in groups:
        E = _phases(ms, n, h).conj().T.contiguous()
        at = torch.from_numpy(first[:, None] + np.arange(n)).to(DEVICE)
        F[:, rows] = (f[:, at.reshape(-1)].reshape(-1, n).to(torch.complex128) @ E
                      ).reshape(B, len(rows), len(ms))
    F = F * weight[None, :, None]
    if spin:
        south, north = F[:, -1, ms.index(spin)].clone(), F[:, 0, ms.index(-spin)].clone()
    F = torch.view_as_real(F.permute(2, 1, 0).contiguous()).reshape(len(ms), len(theta), 2 * B)
    x = torch.zeros((len(ms), L, 2 * B), dtype=torch.float64, device=DEVICE)
    for l0, d in _wigner_d(L, ms, -spin, theta):
        x[:, l0:l0 + d.shape[0]] = torch.bmm(d.permute(1, 0, 2), F)
    x = torch.view_as_complex(x.reshape(len(ms), L, B, 2)).permute(2, 1, 0)
    flm = torch.zeros((B, L, 2 * L - 1), dtype=torch.complex128, device=DEVICE)
    flm[:, :, torch.tensor(ms, device=DEVICE) + L - 1] = x * (
        (-1) ** spin * (_norm(L) if norm is None else norm))[None, :, None]
    if sampling in ("mw", "mwss"):
        # the pole rows' sums run over every l, l < |spin| among them
        # (s2fft/transforms/spherical.py:166-177)
        w = (-1) ** spin * (_norm(L) if norm is None else norm)
        for l in range(abs(spin)):
            flm[:, l, L - 1 + spin] = (-1) ** abs(l - spin) * w[l] * south
            if sampling == "mwss":
                flm[:, l, L - 1 - spin] = w[l] * north
    return _mirror(flm) if reality else flm


def _mirror(flm):
    """The m < 0 half of a real map's coefficients from the m > 0 half."""
    L = flm.shape[1]
    sign = (-1.0) ** torch.arange(1, L, device=DEVICE)
    flm[:, :, :L - 1] = (sign * flm[:, :, L:].conj()).flip(-1)
    return flm


def _generator(seed):
    return torch.Generator(device=DEVICE).manual_seed(int(seed))


def _normal(g, shape, cplx=True):
    re = torch.randn(shape, generator=g, dtype=torch.float64, device=DEVICE)
    return torch.complex(re, torch.randn(shape, generator=g, dtype=torch.float64,
                                         device=DEVICE)) if cplx else re


def _coefficients(g, batch, L, spin, reality):
    """Coefficients with iid normal parts, zero outside |spin|, |m| <= l."""
    flm = _normal(g, (batch, L, 2 * L - 1))
    l = torch.arange(L, device=DEVICE)[:, None]
    m = torch.arange(-(L - 1), L, device=DEVICE)[None, :]
    flm = torch.where((m.abs() <= l) & (l >= abs(spin)), flm, torch.zeros_like(flm))
    if reality:
        flm[:, :, L - 1] = flm[:, :, L - 1].real.to(torch.complex128)
        flm = _mirror(flm)
    return flm


def _pixel_shape(c):
    L = c["L"]
    if c["sampling"] == "healpix":
        return (12 * c["nside"] ** 2,)
    rows = {"mw": L, "mwss": L + 1, "dh": 2 * L, "gl": L}[c["sampling"]]
    return rows, 2 * L if c["sampling"] == "mwss" else 2 * L - 1


def _draws(c, seed):
    """(coefficients, second draw or target): what the case's inputs come from."""
    g = _generator(seed)
    if c["kind"].startswith("wigner"):
        L, N = c["L"], c["N"]
        flmn = torch.cat([_coefficients(g, 1, L, n, False) for n in range(-N + 1, N)])
        return flmn, _normal(g, (2 * N - 1,) + _pixel_shape(c))
    flm = _coefficients(g, c["batch"], c["L"], c["spin"], c["reality"])
    target = None
    if c["kind"] == "forward_gradient":
        target = _coefficients(g, c["batch"], c["L"], c["spin"], c["reality"])
    elif c["kind"] == "inverse_gradient":
        target = _normal(g, (c["batch"],) + _pixel_shape(c), not c["reality"])
    return flm, target


def _wigner_norm(L):
    return (2 * torch.arange(L, device=DEVICE, dtype=torch.float64) + 1) / (8 * math.pi ** 2)


def _wigner_synthesis(flmn, c):
    """sum (2l+1)/8pi^2 flmn d^l_mn e^{i (m alpha + n gamma)}: [gamma, pixel]."""
    N = c["N"]
    planes = torch.cat([(-1) ** n * _synthesis(flmn[N - 1 + n][None], -n, c["sampling"], 0, False,
                                               norm=_wigner_norm(c["L"]))
                        for n in range(-N + 1, N)])
    E = _phases(list(range(-N + 1, N)), 2 * N - 1, 0)  # [n, gamma]
    return E.T.contiguous() @ planes


# ------------------------------------------------------------------ the cases
def prepare(case, seed):
    c = dict(case)
    torch.cuda.set_device(DEVICE)
    kind, L, nside = c["kind"], c["L"], c["nside"] or None
    coef, target = _draws(c, seed)
    state = {"case": c, "coef": coef, "target": target}
    shape = _pixel_shape(c)
    if kind in ("forward", "forward_gradient", "refine", "precompute_forward"):
        f = _synthesis(coef, c["spin"], c["sampling"], c["nside"], c["reality"])
        state["f"] = f.reshape((c["batch"],) + shape)
    elif kind == "wigner_forward":
        state["f"] = _wigner_synthesis(coef, c).reshape((2 * c["N"] - 1,) + shape)
    if kind == "forward_gradient":
        state["f"].requires_grad_(True)
    elif kind in ("inverse_gradient", "wigner_gradient"):
        state["coef"] = coef.requires_grad_(True)
    elif kind == "refine":
        state["network"] = MLPPreconditioner.load(device=DEVICE)
    elif kind == "precompute_forward":
        state["kernel"] = s2fft_amd.precompute_transforms.construct.spin_spherical_kernel(
            L, c["spin"], c["reality"], c["sampling"], nside, True)
    return state


def run(state):
    c = state["case"]
    kind, L, N, spin = c["kind"], c["L"], c["N"], c["spin"]
    sampling, nside, reality = c["sampling"], c["nside"] or None, c["reality"]
    if kind == "forward":
        return s2fft_amd.forward(state["f"], L, spin, nside, sampling, "hip", reality,
                                 iter=c["iter"])
    if kind == "inverse" and c["precision"] == "fp64":
        return s2fft_amd.inverse(state["coef"], L, spin, nside, sampling, "hip", reality)
    if kind == "inverse":
        return sph.inverse_hip(state["coef"], L, spin, nside, sampling, reality,
                               precision=c["precision"])
    if kind == "refine":
        return refine.refine_cg(state["f"], L, spin, nside, sampling, reality, 3,
                                precond=state["network"], learned_steps=1)
    if kind == "forward_gradient":
        flm = s2fft_amd.forward(state["f"], L, spin, nside, sampling, "hip", reality)
        loss = (flm - state["target"]).abs().square().sum()
        return {"flm": flm.detach(), "grad": torch.autograd.grad(loss, state["f"])[0]}
    if kind == "inverse_gradient":
        f = s2fft_amd.inverse(state["coef"], L, spin, nside, sampling, "hip", reality)
        loss = (f - state["target"]).abs().square().sum()
        return {"f": f.detach(), "grad": torch.autograd.grad(loss, state["coef"])[0]}
    if kind == "wigner_forward":
        return s2fft_amd.wigner.forward(state["f"], L, N, None, sampling)
    if kind == "wigner_inverse":
        return s2fft_amd.wigner.inverse(state["coef"], L, N, None, sampling)
    if kind == "wigner_gradient":
        f = s2fft_amd.wigner.inverse(state["coef"], L, N, None, sampling)
        loss = (f - state["target"]).abs().square().sum()
        return {"f": f.detach(), "grad": torch.autograd.grad(loss, state["coef"])[0]}
    return s2fft_amd.precompute_transforms.spherical.forward(
        state["f"], L, spin, state["kernel"], sampling, reality, "hip", nside)


def work(case):
    c = dict(case)
    L, B, real = c["L"], c["batch"], c["reality"]
    wigner = c["kind"].startswith("wigner")
    theta_rows = 4 * c["nside"] - 1 if c["sampling"] == "healpix" else _pixel_shape(c)[0]
    pixels = math.prod(_pixel_shape(c))
    flm = L * (2 * L - 1)
    maps = 2 * c["N"] - 1 if wigner else B
    inout = maps * (16 * flm + (8 if real else 16) * pixels)
    # the recursion (5 flops) and one complex multiply-add per map (4) for every
    # coefficient and ring, rings in pairs for spin 0; a ring's FFT
    coefs = L * (L + 1) // 2 if real else L * L
    rings = theta_rows if wigner or c["spin"] or c["sampling"] == "mw" else (theta_rows + 1) // 2
    one = rings * coefs * (5 + 4) * maps if wigner else rings * coefs * (5 + 4 * B)
    one += maps * 5 * pixels * math.log2(2 * L) * (0.5 if real else 1)
    if c["kind"] == "precompute_forward":
        rows = theta_rows * L * (L if real else 2 * L - 1) * 16
        return {"bytes": inout + rows, "flops": 8 * maps * theta_rows * coefs}
    times = {"refine": 8, "forward_gradient": 2, "inverse_gradient": 2,
             "wigner_gradient": 2}.get(c["kind"], 1 + 2 * c["iter"])
    again = 2 if "gradient" in c["kind"] else 1
    return {"bytes": again * inout, "flops": times * one}


def exact(case, seed):
    c = dict(case)
    torch.cuda.set_device(DEVICE)
    kind, L, spin, real = c["kind"], c["L"], c["spin"], c["reality"]
    sampling, nside, shape = c["sampling"], c["nside"], _pixel_shape(c)
    coef, target = _draws(c, seed)

    def synth(x):
        return _synthesis(x, spin, sampling, nside, real)

    if kind == "wigner_forward":
        return coef
    if kind in ("wigner_inverse", "wigner_gradient"):
        N = c["N"]
        f = _wigner_synthesis(coef, c).reshape((2 * N - 1,) + shape)
        if kind == "wigner_inverse":
            return f
        E = _phases(list(range(-N + 1, N)), 2 * N - 1, 0).conj()
        planes = E @ (2 * (f - target)).reshape(2 * N - 1, -1)
        ones = torch.ones(shape[0], dtype=torch.float64, device=DEVICE)
        grad = torch.cat([(-1) ** n * _projection(planes[N - 1 + n][None], L, -n, sampling, 0, False,
                                                  ones, norm=_wigner_norm(L))
                          for n in range(-N + 1, N)])
        return {"f": f, "grad": grad}
    if kind == "inverse":
        f = synth(coef).reshape((c["batch"],) + shape)
        return f.to(torch.complex128) if sampling == "healpix" else f
    if kind == "inverse_gradient":
        f = synth(coef).reshape((c["batch"],) + shape)
        rows = 4 * nside - 1 if sampling == "healpix" else shape[0]
        ones = torch.ones(rows, dtype=torch.float64, device=DEVICE)
        grad = _projection((2 * (f - target)).reshape(c["batch"], -1), L, spin, sampling, nside,
                           real, ones)
        if real:  # the synthesis reads m >= 0 only and completes the other half
            grad[:, :, :L - 1] = 0
            grad[:, :, L:] *= 2
        return {"f": f.to(torch.complex128) if sampling == "healpix" else f, "grad": grad}
    if kind == "forward_gradient":
        # Gauss-Legendre: the forward's conjugate transpose is the synthesis
        # with the ring weights; real maps: of the Hermitian part of the cotangent
        w = torch.from_numpy(np.polynomial.legendre.leggauss(L)[1][::-1] * 2 * np.pi / (2 * L - 1)
                             ).to(DEVICE)
        grad = _synthesis(2 * (coef - target), spin, sampling, nside, real, ring_weight=w)
        return {"flm": coef, "grad": grad.reshape((c["batch"],) + shape)}
    if kind in ("forward", "precompute_forward") and sampling == "healpix":
        w = torch.full((4 * nside - 1,), 4 * math.pi / (12 * nside * nside), dtype=torch.float64,
                       device=DEVICE)

        def project(f):
            return _projection(f, L, spin, sampling, nside, real, w)

        f = synth(coef)
        flm = project(f)
        for _ in range(c["iter"]):
            flm = flm + project(f - synth(flm))
        return flm
    # sampling theorem, or (refine) the fixed point that the refinement nears
    return coef
