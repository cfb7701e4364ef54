"""Padding rows of the C ABI's ring spectra (needs a GPU): every producer writes
exact zeros into the rows past the grid's (real pairs with a map left over, one and
more launches of the ring FFTs, the VALU and matrix-core syntheses, both layouts) and
nothing past the buffer."""

import pytest
import torch

from s2fft_amd import _lib
from s2fft_amd.sampling import s2_samples
from s2fft_amd.transforms import spherical as sph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sampling,L,nside,reality,batch", [
    ("healpix", 16, 8, True, 1), ("healpix", 18, 9, True, 3), ("healpix", 300, 150, True, 33),
    ("gl", 13, None, False, 2), ("gl", 150, None, False, 17), ("healpix", 16, 8, False, 5),
])
def test_padding_rows_are_zero(sampling, L, nside, reality, batch):
    plan = sph.get_plan(sampling, L, nside, 0, 0, reality)
    lib, st = _lib.lib(), torch.cuda.current_stream().cuda_stream
    rows = s2_samples.ntheta(L, sampling, nside)
    n = lib.s2h_ring_spectra_bytes(plan.handle, batch) // 16
    ncol = L if reality else 2 * L - 1
    pad = n // batch // ncol - rows
    assert 0 < pad < 8

    def buffer():
        return torch.full((n + 64,), float("nan"), dtype=torch.complex128, device="cuda")

    def check(b, tiled=False):
        assert torch.isnan(b[n:].real).all()
        s = b[:n].reshape(batch, -1, ncol, 8).transpose(2, 3).reshape(batch, -1, ncol) if tiled \
            else b[:n].reshape(batch, -1, ncol)
        assert bool((s[:, rows:] == 0).all()) and not torch.isnan(s[:, :rows].real).any()

    f = torch.ones((batch,) + s2_samples.f_shape(L, sampling, nside), device="cuda",
                   dtype=torch.float64 if reality else torch.complex128)
    flm = torch.ones((batch, L, 2 * L - 1), dtype=torch.complex128, device="cuda")
    G, Y, R = buffer(), buffer(), buffer()
    _lib.check(lib.s2h_ring_analysis(plan.handle, f.data_ptr(), int(f.is_complex()), G.data_ptr(),
                                     batch, st))
    check(G)
    for tiled in (False, True) if reality else (False,):
        flags = _lib.SPECTRA_TILED if tiled else 0
        Y.fill_(float("nan"))
        R.fill_(float("nan"))
        _lib.check(lib.s2h_inverse_rings(plan.handle, flm.data_ptr(), Y.data_ptr(), batch,
                                         _lib.PREC_FP64, flags, st))
        check(Y, tiled)
        g = Y if tiled else G
        _lib.check(lib.s2h_ring_residual_ex(plan.handle, g.data_ptr(), Y.data_ptr(), None,
                                            R.data_ptr(), None, None, batch, flags, st))
        check(R, tiled)
