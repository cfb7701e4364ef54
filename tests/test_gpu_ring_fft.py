"""The ring FFT kernels (s2h_ring_fft.hip) at every transform size they have,
against numpy's FFT of each ring: convolutions of 64 to 8192 points, powers of
two of 64 to 4096, the grid in one launch (few workgroups) and in one per size
(many), real pairs with an odd map left over; needs a GPU.

Tolerance: two transforms of up to 8192 points and two chirp products per value
round by a few eps each per pass; 1e-12 of the largest value holds an order of
magnitude beyond that."""

import numpy as np
import pytest
import torch

from oracle import ffts as offts, geometry as geo
from tests.conftest import max_rel

from s2fft_amd import _lib
from s2fft_amd.transforms import spherical as sph

pytestmark = pytest.mark.gpu
TOL = 1e-12


def _stream():
    return torch.cuda.current_stream().cuda_stream


# nside 3 .. 1024: belts of 12, 64, 400, 512, 1024, 2400 and 4096 pixels
@pytest.mark.parametrize("nside,L,batch", [(1, 2, 1), (3, 8, 2), (16, 32, 1), (100, 211, 1),
                                           (128, 256, 3), (256, 512, 1), (600, 1200, 1),
                                           (1024, 2048, 1), (64, 130, 70)])
def test_complex_rings_both_directions(nside, L, batch):
    rng = np.random.default_rng(nside)
    f = rng.standard_normal((batch, 12 * nside**2)) + 1j * rng.standard_normal(
        (batch, 12 * nside**2))
    ft = torch.from_numpy(f).cuda()
    out = torch.empty((batch, 4 * nside - 1, 2 * L), dtype=torch.complex128, device="cuda")
    lib = _lib.lib()
    _lib.check(lib.s2h_healpix_fft_prepare(nside, L))
    _lib.check(lib.s2h_healpix_fft(nside, L, 0, ft.data_ptr(), out.data_ptr(), batch, _stream()))
    for b in {0, batch - 1}:
        assert max_rel(out[b].cpu().numpy(), offts.healpix_fft(f[b], L, nside)) < TOL
    back = torch.empty_like(ft)
    spec = rng.standard_normal(out.shape) + 1j * rng.standard_normal(out.shape)
    st = torch.from_numpy(spec).cuda()
    _lib.check(lib.s2h_healpix_ifft(nside, L, 0, st.data_ptr(), back.data_ptr(), batch, _stream()))
    for b in {0, batch - 1}:
        assert max_rel(back[b].cpu().numpy(), offts.healpix_ifft(spec[b], L, nside)) < TOL


def _ring_spectra(f, L, nside):
    """w e^{-i m phi0} DFT of every ring of a real map, m in [0, L)."""
    offs, n = offts.ring_offsets(nside)
    phi0 = geo.healpix_phi0(np.arange(4 * nside - 1), nside)
    m = np.arange(L)
    rows = [np.fft.fft(f[o:o + k])[m % k] * np.exp(-1j * m * p) for o, k, p in zip(offs, n, phi0)]
    return np.array(rows) * 4 * np.pi / (12 * nside**2)


@pytest.mark.parametrize("nside,L,batch", [(16, 32, 3), (24, 61, 1), (128, 256, 5), (192, 449, 2),
                                           (256, 700, 3)])
def test_real_rings_in_pairs(nside, L, batch):
    """L = 700 at nside 256 has more columns than half the belt's pixels."""
    rng = np.random.default_rng(L)
    f = rng.standard_normal((batch, 12 * nside**2))
    plan = sph.get_plan("healpix", L, nside, 0, 0, True)
    G = sph.ring_analysis_hip(torch.from_numpy(f).cuda(), plan).cpu().numpy()
    for b in range(batch):
        got = G[b].reshape(-1, L)[:4 * nside - 1]
        assert max_rel(got, _ring_spectra(f[b], L, nside)) < TOL


@pytest.mark.parametrize("nside,L", [(16, 32), (100, 230), (256, 512)])
def test_real_synthesis_in_pairs(nside, L):
    """Three real maps in one call, as float64 and as complex128, and their
    residual, against the maps one by one as the transform of complex maps."""
    g = torch.Generator(device="cuda").manual_seed(L)
    re, im = (torch.randn((3, L, 2 * L - 1), generator=g, dtype=torch.float64, device="cuda")
              for _ in range(2))
    l, m = torch.arange(L, device="cuda")[:, None], torch.arange(2 * L - 1, device="cuda") - L + 1
    flm = torch.where((m >= 0) & (m <= l), torch.complex(re, torch.where(m == 0, 0.0, im)), 0.0)
    sign = (-1.0) ** torch.arange(1, L, device="cuda")
    flm[:, :, :L - 1] = (sign * flm[:, :, L:].conj()).flip(-1)
    want = torch.cat([sph.inverse_hip(flm[b:b + 1], L, 0, nside, "healpix", False)
                      for b in range(3)]).real
    real = sph.inverse_hip(flm, L, 0, nside, "healpix", True, real_output=True)
    cplx = sph.inverse_hip(flm, L, 0, nside, "healpix", True)
    sub = torch.randn(cplx.shape, generator=g, dtype=torch.float64, device="cuda") * (1 + 2j)
    left = sph.inverse_hip(flm, L, 0, nside, "healpix", True, sub_from=sub.clone())
    assert real.dtype == torch.float64 and max_rel(real.cpu(), want.cpu()) < TOL
    assert bool((cplx.imag == 0).all()) and max_rel(cplx.real.cpu(), want.cpu()) < TOL
    assert max_rel((sub - left).cpu(), want.cpu()) < TOL


@pytest.mark.parametrize("sampling,L", [("mwss", 8), ("mwss", 32), ("mwss", 64), ("mwss", 128),
                                        ("mwss", 256), ("gl", 16), ("gl", 33), ("gl", 128),
                                        ("gl", 129)])
def test_equiangular_round_trip(sampling, L):
    """One length per grid: 16 to 512 points as powers of two or not, 31 to 257."""
    g = torch.Generator(device="cuda").manual_seed(L)
    flm = torch.randn((2, L, 2 * L - 1), generator=g, dtype=torch.complex128, device="cuda")
    l, m = torch.arange(L, device="cuda")[:, None], torch.arange(2 * L - 1, device="cuda") - L + 1
    flm = torch.where(m.abs() <= l, flm, 0.0)
    f = sph.inverse_hip(flm, L, 0, None, sampling)
    assert max_rel(sph.forward_hip(f, L, 0, None, sampling).cpu(), flm.cpu()) < 1e-11
