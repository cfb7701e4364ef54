"""The latitudinal kernels of small batches against those of larger ones (needs a GPU).

Batches of 1 to 3 maps take the VALU kernels, larger ones at the larger sizes the
matrix-core projection: the same maps alone and inside a batch of 5 have to agree.  The sizes cover one and
several waves of rings, one to eight rings per lane, last waves of one ring, pairs
with and without an equator, pole rows (also for l < |spin|), a first l above zero,
and the most rings a plan has (4096).  Both sides carry
FP64 rounding of about 1e-13 at these band-limits; a wrong ring, row or order is an
error of order one.
"""

import pytest
import torch

import s2fft_amd
from s2fft_amd.sampling import s2_samples

pytestmark = pytest.mark.gpu
TOL = 1e-12

CASES = [
    # sampling, L, nside, spin, reality, L_lower
    ("mw", 2, None, 0, False, 0),
    ("mw", 5, None, 3, False, 0),
    ("mw", 65, None, -2, False, 0),
    ("mwss", 64, None, 0, True, 0),
    ("mwss", 129, None, 1, False, 5),
    ("gl", 128, None, 0, True, 0),
    ("gl", 131, None, 2, False, 7),
    ("dh", 259, None, 1, False, 0),
    ("mw", 520, None, 0, False, 0),
    ("gl", 700, None, 0, False, 0),
    ("healpix", 35, 17, 0, True, 0),
    ("healpix", 600, 300, 1, False, 0),
    ("dh", 2048, None, 1, False, 0),
]


def _flm(L, B, reality, gen):
    flm = torch.randn(B, L, 2 * L - 1, 2, generator=gen, dtype=torch.float64)
    flm = torch.view_as_complex(flm)
    el = torch.arange(L)[:, None]
    m = torch.arange(-(L - 1), L)[None, :]
    flm = flm * (m.abs() <= el)
    if reality:
        sign = 1.0 - 2.0 * (m % 2)
        flm = 0.5 * (flm + sign * flm.flip(-1).conj())
    return flm.cuda()


def _rel(a, b):
    return float((a - b).abs().max() / b.abs().max().clamp_min(1e-300))


@pytest.mark.parametrize("sampling,L,nside,spin,reality,lower", CASES)
def test_small_batches_match_larger(sampling, L, nside, spin, reality, lower):
    gen = torch.Generator().manual_seed(L + 3)
    kw = dict(spin=spin, nside=nside, sampling=sampling, reality=reality, L_lower=lower)
    flm = _flm(L, 5, reality, gen)
    f = s2fft_amd.inverse(flm, L, **kw)
    back = s2fft_amd.forward(f, L, **kw)
    for n in (1, 2, 3):
        assert _rel(s2fft_amd.inverse(flm[:n], L, **kw), f[:n]) < TOL
        assert _rel(s2fft_amd.forward(f[:n], L, **kw), back[:n]) < TOL


@pytest.mark.parametrize("sampling,L,nside,spin,reality", [
    ("healpix", 24, 12, 0, True), ("healpix", 19, 9, 1, False), ("healpix", 1030, 515, 1, False),
])
def test_accumulating_forward(sampling, L, nside, spin, reality):
    gen = torch.Generator().manual_seed(L)
    f = torch.randn((5,) + s2_samples.f_shape(L, sampling, nside), generator=gen,
                    dtype=torch.float64 if reality else torch.complex128).cuda()
    kw = dict(spin=spin, nside=nside, sampling=sampling, reality=reality, iter=2)
    ref = s2fft_amd.forward(f, L, **kw)
    for n in (1, 3):
        assert _rel(s2fft_amd.forward(f[:n], L, **kw), ref[:n]) < TOL


@pytest.mark.parametrize("sampling,L,nside,spin,reality", [
    ("mw", 67, None, 2, False), ("mwss", 130, None, 0, True), ("gl", 600, None, 0, False),
    ("healpix", 140, 70, 1, False),
])
def test_gradients_are_the_adjoints(sampling, L, nside, spin, reality):
    # <g, A x> against <A^H g, x> with A applied to a batch of 5
    gen = torch.Generator().manual_seed(L)
    kw = dict(spin=spin, nside=nside, sampling=sampling, reality=reality)
    flm = _flm(L, 5, reality, gen).requires_grad_()
    f = s2fft_amd.inverse(flm, L, **kw)
    g = torch.randn(f.shape, generator=gen, dtype=f.dtype).cuda()
    lhs = float((g.conj() * f).real.sum())
    (gx,) = torch.autograd.grad(f, flm, g)
    assert abs(float((gx.conj() * flm).real.sum()) - lhs) < TOL * float(g.norm() * f.norm())
    x = f.detach().requires_grad_()
    out = s2fft_amd.forward(x, L, **kw)
    h = _flm(L, 5, False, gen)
    lhs = float((h.conj() * out).real.sum())
    (gf,) = torch.autograd.grad(out, x, h)
    assert abs(float((gf.conj() * x).real.sum()) - lhs) < TOL * float(h.norm() * out.norm())
