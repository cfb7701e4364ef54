"""The error of MW / MWSS forwards in reduced precision (needs a GPU).

A coefficient is a sum over rings of rounded d times rounded rows.  The roundings are
independent, so that 2N rows leave 1 / sqrt 2 of the error of N rows (the terms are half
as large).  Relative RMS over random coefficients, measured with the 2L + 1 rows of MWSS
at 2L: single BF16 1.53e-3, split BF16 2.9e-6 at every L; with L + 1 rows 2.16e-3 and
4.1e-6.  The bounds lie between the two.  FP32 adds the accumulation, which grows with
the rings of a chain: 5.4e-8 at L = 24 to 1.77e-7 at L = 1024 with 2L + 1 rows and 128
rings per chain; the bounds are those errors.
"""

import pytest
import torch

from s2fft_amd.transforms import spherical as sph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sampling", ["mw", "mwss"])
@pytest.mark.parametrize("L,batch,spin,reality,mixed", [
    (24, 8, 0, False, 5.5e-8), (64, 8, 2, False, 1.2e-7), (101, 8, 0, True, 1.0e-7),
    (256, 4, 2, False, 1.58e-7), (385, 4, 0, False, 1.42e-7), (385, 4, 0, True, 1.42e-7),
    (512, 8, -1, False, 1.7e-7), (1024, 1, 0, False, 1.77e-7),
])
def test_rms_error(sampling, L, batch, spin, reality, mixed):
    gen = torch.Generator().manual_seed(L)
    flm = torch.randn((batch, L, 2 * L - 1), generator=gen, dtype=torch.complex128)
    m, l = torch.arange(-(L - 1), L)[None, :], torch.arange(L)[:, None]
    flm = flm * ((m.abs() <= l) & (l >= abs(spin)))
    if reality:
        flm = 0.5 * (flm + (1.0 - 2.0 * (m % 2)) * flm.flip(-1).conj())
    flm = flm.cuda()
    f = sph.inverse_hip(flm, L, spin, None, sampling, reality)
    for precision, bound in (("bf16x1", 1.8e-3), ("bf16", 3.4e-6), ("mixed", mixed)):
        got = sph.forward_hip(f, L, spin, None, sampling, reality, precision=precision)
        assert float((got - flm).norm() / flm.norm()) < bound, precision


@pytest.mark.parametrize("sampling", ["mw", "mwss"])
@pytest.mark.parametrize("L,batch,spin,reality", [(2, 3, 1, False), (17, 2, -1, False),
                                                  (64, 1, 0, False), (65, 64, 2, False),
                                                  (130, 2, 0, True), (512, 8, 1, False)])
def test_noise_maps(sampling, L, batch, spin, reality):
    """Maps that are not band-limited: the theta-Nyquist term and the pole samples take
    part, and every tile choice of the product.  White noise has as much outside the band
    as inside: twice the split-BF16 error, 1e-5 of the RMS with room; a term left out
    shows at 1 / L or more."""
    gen = torch.Generator().manual_seed(L)
    shape = (batch,) + sph.samples.f_shape(L, sampling, None)
    f = torch.randn(shape, generator=gen, dtype=torch.float64 if reality
                    else torch.complex128).cuda()
    want = sph.forward_hip(f, L, spin, None, sampling, reality)
    got = sph.forward_hip(f, L, spin, None, sampling, reality, precision="bf16")
    assert float((got - want).norm() / want.norm()) < 1e-5
