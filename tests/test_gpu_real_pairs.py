"""Batches of real maps against each map alone, for coefficients as an optimisation
hands them over: the imaginary part at m = 0 not zero (needs a GPU).

Real rings are transformed in pairs x + i y.  A map alone has no imaginary part at m =
0 (it takes the real part of the sum), so inside a batch it has to have none either.  Maps returned as complex128 are
transformed alone: a partner that is larger by 1e8 or holds a NaN leaves no trace.
FP64 rounding of two maps of one scale: 1e-13 of a map's own maximum is some hundred
eps; the imaginary parts are of order one.
"""

import pytest
import torch

import s2fft_amd
from s2fft_amd import precompute_transforms as pc
from s2fft_amd.transforms import spherical as sph

pytestmark = pytest.mark.gpu
TOL = 1e-13


def _flm(B, L, seed):
    gen = torch.Generator().manual_seed(seed)
    flm = torch.randn((B, L, 2 * L - 1), generator=gen, dtype=torch.complex128)
    m = torch.arange(-(L - 1), L)[None, :]
    return (flm * (m.abs() <= torch.arange(L)[:, None])).cuda()


def _own_error(got, want):
    return float((got - want).abs().max() / want.abs().max())


@pytest.mark.parametrize("sampling,L,nside", [("healpix", 16, 8), ("healpix", 61, 30),
                                              ("gl", 20, None), ("mw", 33, None),
                                              ("mwss", 32, None), ("dh", 17, None)])
@pytest.mark.parametrize("batch", [2, 3, 9])
def test_m0_stays_with_its_map(sampling, L, nside, batch):
    flm = _flm(batch, L, L)
    kw = dict(nside=nside, sampling=sampling, reality=True)
    for real_output in (False, True):
        got = sph.inverse_hip(flm, L, real_output=real_output, **kw)
        for b in range(batch):
            one = sph.inverse_hip(flm[b:b + 1], L, real_output=real_output, **kw)[0]
            assert _own_error(got[b], one) < TOL
    # and the gradient says the same
    x = flm.clone().requires_grad_()
    g = torch.randn(s2fft_amd.inverse(flm, L, **kw).shape, dtype=torch.float64,
                    generator=torch.Generator("cuda").manual_seed(1), device="cuda")
    (grad,) = torch.autograd.grad(s2fft_amd.inverse(x, L, **kw).real, x, g)
    for b in range(batch):
        x = flm[b].clone().requires_grad_()
        (one,) = torch.autograd.grad(s2fft_amd.inverse(x, L, **kw).real, x, g[b])
        assert _own_error(grad[b], one) < TOL


@pytest.mark.parametrize("sampling,L,nside", [("healpix", 16, 8), ("gl", 20, None)])
def test_m0_stays_with_its_map_stored_kernel(sampling, L, nside):
    flm = _flm(3, L, L)
    kw = dict(nside=nside, sampling=sampling, reality=True)
    got = pc.spherical.inverse(flm, L, **kw)
    for b in range(3):
        assert _own_error(got[b], pc.spherical.inverse(flm[b], L, **kw)) < TOL


@pytest.mark.parametrize("L,nside", [(16, 8), (61, 30), (200, 100), (256, 128)])
def test_complex_maps_are_alone(L, nside):
    flm = _flm(3, L, L)
    flm[1] *= 1e8
    nan = flm.clone()
    nan[1, 3, L] = float("nan")
    kernel = pc.construct.spin_spherical_kernel(L, 0, True, "healpix", nside, False) \
        if L < 100 else None
    calls = [lambda x: sph.inverse_hip(x, L, 0, nside, "healpix", True)]
    if kernel is not None:
        calls.append(lambda x: pc.spherical.inverse(x, L, 0, kernel, "healpix", True, nside=nside))
    for call in calls:
        one = [call(flm[b:b + 1])[0] for b in range(3)]
        got, with_nan = call(flm), call(nan)
        for b in range(3):
            assert _own_error(got[b], one[b]) < TOL
        for b in (0, 2):
            assert _own_error(with_nan[b], one[b]) < TOL


@pytest.mark.parametrize("sampling,L,nside", [
    *(("gl", L, None) for L in (9, 30, 50, 100, 200, 400, 900, 1500)),
    *(("mwss", L, None) for L in (4, 8, 16, 32, 64, 128, 256, 512, 1024, 2048)),
    *(("healpix", L, n) for L, n in ((40, 17), (150, 64), (211, 100), (230, 100), (300, 128),
                                     (700, 300), (1100, 512), (1300, 600), (2100, 1024))),
])
def test_pairs_at_every_transform_size(sampling, L, nside):
    """Three real maps in both directions against the complex transform of each alone:
    convolutions of 64 to 8192 points, powers of two of 8 to 4096, and ragged grids of
    them.  Pixels within 1e-12 of the maximum; coefficients by their RMS, 1e-12 too (their
    largest differences sit at l = L - 1, |m| <= 2, where the forward is conditioned
    worst: 2e-12 to 6e-12 at L = 2048 with any ring transform, at 1e-14 of RMS)."""
    flm = _flm(3, L, L)
    m = torch.arange(-(L - 1), L, device="cuda")
    flm = 0.5 * (flm + (1.0 - 2.0 * (m % 2)) * flm.flip(-1).conj())
    want = torch.cat([sph.inverse_hip(flm[b:b + 1], L, 0, nside, sampling, False)
                      for b in range(3)]).real.contiguous()
    got = sph.inverse_hip(flm, L, 0, nside, sampling, True, real_output=True)
    assert _own_error(got, want) < 1e-12
    alone = sph.inverse_hip(flm, L, 0, nside, sampling, True)
    assert _own_error(alone.real if alone.is_complex() else alone, want) < 1e-12
    got = sph.forward_hip(want, L, 0, nside, sampling, True)
    for b in range(3):
        one = sph.forward_hip(want[b:b + 1].to(torch.complex128), L, 0, nside, sampling, False)[0]
        assert float((got[b] - one).norm() / one.norm()) < 1e-12
