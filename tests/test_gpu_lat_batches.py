"""Which kernels a batch of FP64 transforms takes (needs a GPU).

A batch of any size has to hold what each of its maps gives alone (the VALU kernels):
4, 8 and 9 maps (the limit of the VALU inverse), 16 (one tile of the matrix-core
inverse), 17 and 24 (a tile and the rest), 26 (two tiles).  The smaller band-limits
stay on the VALU kernels throughout, the larger ones pass both limits.  FP64 rounding
of about 1e-13 at these sizes; a wrong map or row is an error of order one.
"""

import pytest
import torch

import s2fft_amd

pytestmark = pytest.mark.gpu
TOL = 1e-12


@pytest.mark.parametrize("sampling,L,nside,spin,reality", [
    ("mw", 20, None, 1, False), ("mw", 130, None, -2, False), ("mwss", 130, None, 0, False),
    ("gl", 190, None, 0, True), ("dh", 100, None, 2, False), ("healpix", 193, 96, 0, True),
])
def test_batches_match_single_maps(sampling, L, nside, spin, reality):
    gen = torch.Generator().manual_seed(L)
    n = 26
    flm = torch.randn((n, L, 2 * L - 1), generator=gen, dtype=torch.complex128)
    m = torch.arange(-(L - 1), L)[None, :]
    flm = flm * (m.abs() <= torch.arange(L)[:, None])
    if reality:
        flm = 0.5 * (flm + (1.0 - 2.0 * (m % 2)) * flm.flip(-1).conj())
    flm = flm.cuda()
    kw = dict(spin=spin, nside=nside, sampling=sampling, reality=reality)
    f = torch.stack([s2fft_amd.inverse(flm[b], L, **kw) for b in range(n)])
    back = torch.stack([s2fft_amd.forward(f[b], L, **kw) for b in range(n)])
    for b in (4, 8, 9, 16, 17, 24, 26):
        got = s2fft_amd.inverse(flm[:b], L, **kw)
        assert float((got - f[:b]).abs().max()) < TOL * float(f.abs().max())
        got = s2fft_amd.forward(f[:b], L, **kw)
        assert float((got - back[:b]).abs().max()) < TOL * float(back.abs().max())
