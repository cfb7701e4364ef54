"""Batches that fill the card against their maps alone (needs a GPU).

The theta operators through LDS (from 4096 waves on: row and column blocks that are
not full, real and complex signals, the theta-Nyquist term of MWSS, forward and
adjoint), and the FP64 matrix-core projection of 16-map tiles with one set of pairs
on 4 waves (up to 256 pairs), on 8 waves (more) and two passes (more than 512).  FP64
rounding of about 1e-13 at these sizes; a wrong row, column or map is an error of
order one.
"""

import pytest
import torch

import s2fft_amd
from s2fft_amd.sampling import s2_samples

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("sampling,L,nside,spin,reality,batch", [
    ("mw", 70, None, 1, False, 208), ("mwss", 70, None, -2, False, 208),
    ("mw", 131, None, 0, True, 150), ("mwss", 65, None, 0, True, 700),
    ("gl", 150, None, 0, True, 100), ("gl", 530, None, 0, True, 12),
    ("healpix", 530, 262, 0, True, 9),
])
def test_forward_and_gradient(sampling, L, nside, spin, reality, batch):
    gen = torch.Generator().manual_seed(L)
    kw = dict(spin=spin, nside=nside, sampling=sampling, reality=reality)
    f = torch.randn((batch,) + s2_samples.f_shape(L, sampling, nside), generator=gen,
                    dtype=torch.float64 if reality else torch.complex128).cuda()
    g = torch.randn((batch, L, 2 * L - 1), generator=gen, dtype=torch.complex128).cuda()
    x = f.clone().requires_grad_()
    out = s2fft_amd.forward(x, L, **kw)
    (grad,) = torch.autograd.grad(out, x, g)
    out = out.detach()
    for b in (0, 1, batch // 2, batch - 1):
        x = f[b].clone().requires_grad_()
        ref = s2fft_amd.forward(x, L, **kw)
        assert float((out[b] - ref.detach()).abs().max()) < TOL * float(ref.detach().abs().max())
        (ref,) = torch.autograd.grad(ref, x, g[b])
        assert float((grad[b] - ref).abs().max()) < TOL * float(ref.abs().max())
