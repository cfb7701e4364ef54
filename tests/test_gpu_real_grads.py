"""Gradients of batched real forwards for cotangents that are not conjugate-
symmetric (needs a GPU): the ring transforms take real maps in pairs, and the
gradient of a map alone and inside a batch has to be the same (FP64 rounding:
1e-13 of the largest value holds many eps at L = 12)."""

import pytest
import torch

import s2fft_amd
from s2fft_amd.sampling import s2_samples

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sampling,L,nside", [("gl", 12, None), ("mw", 7, None),
                                              ("mwss", 8, None), ("healpix", 16, 8)])
def test_pairs_do_not_mix(sampling, L, nside):
    gen = torch.Generator().manual_seed(L)
    f = torch.randn((3,) + s2_samples.f_shape(L, sampling, nside), generator=gen,
                    dtype=torch.float64).cuda()
    h = torch.randn((3, L, 2 * L - 1), generator=gen, dtype=torch.complex128).cuda()

    def grad(x, g):
        x = x.clone().requires_grad_()
        out = s2fft_amd.forward(x, L, nside=nside, sampling=sampling, reality=True)
        return torch.autograd.grad(out, x, g)[0]

    got = grad(f, h)
    for b in range(3):
        one = grad(f[b:b + 1], h[b:b + 1])[0]
        assert float((got[b] - one).abs().max()) < 1e-13 * float(one.abs().max())
