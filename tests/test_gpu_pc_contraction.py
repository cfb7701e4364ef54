"""The contraction of the precompute path with an arbitrary stored kernel, against
numpy's FFT of each ring and einsum (needs a GPU): rows, steps and m that do not
fill their tiles, few steps, batches of every chunk size with remainders, real and
complex kernels, entries at l < |m| that are not zero, both directions.  A sum of
up to 67 terms and one FFT of up to 133 points in FP64: 1e-13 of the largest value
is some hundred eps."""

import numpy as np
import pytest
import torch

from s2fft_amd.precompute_transforms import spherical as pspin

pytestmark = pytest.mark.gpu
TOL = 1e-13


@pytest.mark.parametrize("L,batch,reality,kernel_complex", [
    (2, 1, False, False), (3, 2, True, False), (8, 1, False, True), (16, 4, False, False),
    (17, 3, True, True), (33, 5, False, True), (50, 9, True, False), (67, 2, False, False),
    (64, 16, True, True),
])
def test_random_kernel(L, batch, reality, kernel_complex):
    rng = np.random.default_rng(L)
    n, nm = 2 * L - 1, L if reality else 2 * L - 1
    m = np.arange(0 if reality else -(L - 1), L)
    K = rng.standard_normal((L, L, nm))
    if kernel_complex:
        K = K + 1j * rng.standard_normal(K.shape) * (m > 0 if reality else 1)  # real at m = 0
    f = rng.standard_normal((batch, L, n))
    if not reality:
        f = f + 1j * rng.standard_normal(f.shape)
    kt = torch.from_numpy(K).cuda()
    got = pspin.forward(torch.from_numpy(f).cuda(), L, 0, kt, "gl", reality).cpu().numpy()
    spec = np.fft.fft(f, axis=-1)[:, :, m % n]
    ref = np.einsum("tlm,btm->blm", K, spec)
    assert np.max(np.abs(got[:, :, L - 1 + m] - ref)) < TOL * np.max(np.abs(ref))
    if reality:
        sign = (-1.0) ** m[1:]
        assert np.array_equal(got[:, :, L - 1 - m[1:]], sign * got[:, :, L - 1 + m[1:]].conj())

    flm = rng.standard_normal((batch, L, n)) + 1j * rng.standard_normal((batch, L, n))
    if reality:
        flm[:, :, L - 1] = flm[:, :, L - 1].real
    f = pspin.inverse(torch.from_numpy(flm).cuda(), L, 0, kt, "gl", reality).cpu().numpy()
    rows = np.einsum("tlm,blm->btm", K, flm[:, :, L - 1 + m])
    phase = np.exp(2j * np.pi * np.outer(m, np.arange(n)) / n)
    if reality:
        ref = 2 * np.real(rows @ phase) - rows[:, :, :1].real
    else:
        ref = rows @ phase
    assert np.max(np.abs(f - ref)) < TOL * np.max(np.abs(ref))
