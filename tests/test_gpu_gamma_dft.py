"""The gamma DFT at every N it has, in its six modes, with one output per thread (few
samples, a last block not full) and all of them (many), against sums in numpy (needs a
GPU).  At most 15 terms in FP64: 1e-14 of the largest value is some tens of eps."""

import numpy as np
import pytest
import torch

from s2fft_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npix", [300, 140000])
@pytest.mark.parametrize("N", range(1, 9))
def test_modes(N, npix):
    G, lib, st = 2 * N - 1, _lib.lib(), torch.cuda.current_stream().cuda_stream
    rng = np.random.default_rng(N)
    real = rng.standard_normal((G, npix))
    cplx = real + 1j * rng.standard_normal((G, npix))
    n, g = np.arange(-(N - 1), N), np.arange(G)
    E = np.exp(2j * np.pi * np.outer(n, g) / G)  # [n][g]
    half = np.where(np.arange(N) > 0, 2.0, 1.0)[:, None]
    want = {0: E.conj() @ cplx, 2: E.conj() @ real, 1: E.T @ cplx,
            3: np.real(E[N - 1:].T @ (half * cplx[:N])), 4: np.real(E[N - 1:].T @ cplx[:N]),
            5: half * (E[N - 1:].conj() @ real)}
    for mode, ref in want.items():
        src = torch.from_numpy({2: real, 5: real, 3: cplx[:N], 4: cplx[:N]}.get(mode, cplx)).cuda()
        out = torch.full(ref.shape, float("nan"), device="cuda",
                         dtype=torch.complex128 if np.iscomplexobj(ref) else torch.float64)
        _lib.check(lib.s2h_gamma_dft(N, npix, mode, 0.5, src.contiguous().data_ptr(),
                                     out.data_ptr(), st))
        ref = 0.5 * ref
        assert np.max(np.abs(out.cpu().numpy() - ref)) < 1e-14 * np.max(np.abs(ref)), mode
