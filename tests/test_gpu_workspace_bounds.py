"""No call writes past s2h_workspace_bytes (needs a GPU): the bytes after it, in the same
allocation, stay as they were.  The smallest band-limits, where rows padded to whole
blocks weigh most, and sizes around a block of 8 rows."""

import pytest
import torch

from s2fft_amd import _lib
from s2fft_amd.sampling import s2_samples
from s2fft_amd.transforms import spherical as sph

pytestmark = pytest.mark.gpu
TAIL = 1 << 16


@pytest.mark.parametrize("reality", [False, True])
@pytest.mark.parametrize("L", [2, 3, 4, 7, 8, 9, 16])
@pytest.mark.parametrize("sampling", ["mw", "mwss", "gl", "dh", "healpix"])
def test_tail_of_the_workspace_is_untouched(sampling, L, reality):
    nside = L // 2 if sampling == "healpix" else None
    plan = sph.get_plan(sampling, L, nside, 0, 0, reality)
    lib, st = _lib.lib(), torch.cuda.current_stream().cuda_stream
    for batch in (1, 2, 5):
        n = plan.workspace_bytes(batch)
        work = torch.full((n + TAIL,), 0xA5, dtype=torch.uint8, device="cuda")
        f = torch.ones((batch,) + s2_samples.f_shape(L, sampling, nside), device="cuda",
                       dtype=torch.float64 if reality else torch.complex128)
        out = torch.empty(f.shape, device="cuda", dtype=torch.complex128)
        flm = torch.ones((batch, L, 2 * L - 1), dtype=torch.complex128, device="cuda")
        _lib.check(lib.s2h_forward(plan.handle, f.data_ptr(), int(f.is_complex()),
                                   flm.data_ptr(), work.data_ptr(), batch, st))
        _lib.check(lib.s2h_forward_adjoint(plan.handle, flm.data_ptr(), out.data_ptr(),
                                           work.data_ptr(), batch, st))
        _lib.check(lib.s2h_inverse(plan.handle, flm.data_ptr(), out.data_ptr(), work.data_ptr(),
                                   batch, st))
        _lib.check(lib.s2h_inverse_adjoint(plan.handle, f.data_ptr(), int(f.is_complex()),
                                           flm.data_ptr(), work.data_ptr(), batch, st))
        assert bool((work[n:] == 0xA5).all()), batch
