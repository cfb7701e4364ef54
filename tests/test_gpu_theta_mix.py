"""The theta operators of the MW / MWSS forward (s2h_theta_mix.hip) on maps that
are not band-limited (white noise: every harmonic, the theta-Nyquist term and the
pole samples of odd columns take part), against the oracle's resampling chain,
at tile edges and for every tile choice; needs a GPU.

Tolerance: the oracle's m-recursion drifts by 4.5e-12 at L = 256
(tests/test_oracle_pins.py), the operators' products round like sqrt(L) eps:
1e-11 for L <= 130 with margin for the noise maps' larger rows."""

import numpy as np
import pytest
import torch

from oracle import geometry as geo, transforms as otr
from tests.conftest import max_rel

import s2fft_amd
from s2fft_amd.transforms import spherical as sph

pytestmark = pytest.mark.gpu
TOL = 1e-11


def _noise(L, sampling, batch, reality, seed):
    rng = np.random.default_rng(seed)
    shape = (batch,) + geo.f_shape(L, sampling)
    f = rng.standard_normal(shape)
    return f if reality else f + 1j * rng.standard_normal(shape)


@pytest.mark.parametrize("sampling", ["mw", "mwss"])
@pytest.mark.parametrize("L,spin,reality", [(2, 0, False), (3, 1, False), (15, 0, True),
                                            (16, 2, False), (17, -1, False), (64, 0, False),
                                            (65, -2, False), (129, 1, False), (130, 0, True)])
def test_noise_maps_match_the_resampling_chain(sampling, L, spin, reality):
    f = _noise(L, sampling, 1, reality, L + 7 * spin)
    got = s2fft_amd.forward(f[0], L, spin, None, sampling, "hip", reality)
    assert max_rel(got, otr.forward(f[0], L, spin, None, sampling, reality)) < TOL


@pytest.mark.parametrize("sampling,L,spin,batch", [("mw", 65, 2, 64), ("mwss", 65, 1, 64),
                                                   ("mw", 47, -1, 140)])
def test_larger_tiles_agree_with_the_smallest(sampling, L, spin, batch):
    """These batches take the 2 x 2 tiles, single maps 1 x 1."""
    f = _noise(L, sampling, batch, False, 11)
    got = s2fft_amd.forward(torch.from_numpy(f).cuda(), L, spin, None, sampling).cpu().numpy()
    for b in (0, 1, batch - 1):
        assert max_rel(got[b], s2fft_amd.forward(f[b], L, spin, None, sampling)) < 1e-13
    assert max_rel(got[batch // 2], otr.forward(f[batch // 2], L, spin, None, sampling)) < TOL


@pytest.mark.parametrize("sampling", ["mw", "mwss"])
@pytest.mark.parametrize("L,spin", [(2, 0), (16, 1), (33, -2), (65, 0)])
def test_adjoint_identity_on_noise(sampling, L, spin):
    """<y, F x> = <F^H y, x> with F from the oracle."""
    rng = np.random.default_rng(L)
    x = _noise(L, sampling, 1, False, 3 * L)[0]
    y = rng.standard_normal((L, 2 * L - 1)) + 1j * rng.standard_normal((L, 2 * L - 1))
    lhs = np.vdot(y, otr.forward(x, L, spin, None, sampling))
    fhy = sph.forward_adjoint_hip(torch.from_numpy(y)[None].cuda(), L, spin, None, sampling)[0]
    rhs = np.vdot(fhy.cpu().numpy(), x)
    assert abs(lhs - rhs) < TOL * np.linalg.norm(x) * np.linalg.norm(y)
