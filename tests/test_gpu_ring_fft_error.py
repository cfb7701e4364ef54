"""RMS error of the ring FFTs by kind and length of ring, against numpy's in extended
precision (needs a GPU).

The bounds are what transforms in passes through LDS left (radix 8, with the odd primes
up to 13, convolutions for the other lengths), measured over the same kinds of rings:
powers of two 2.6e-16 up to 256 points, 3.5e-16 up to 1024 and 4.5e-16 above, and below
64 points 1.2e-16 forward and 2.8e-16 back, whose folding of the spectrum adds its own;
other rings 4.9e-16 below 64 points (12, 20, 28, 44 and 52, the most accurate ones),
6.6e-16 up to 400, 7.3e-16 up to 1100 and 8.3e-16 above.  An RMS over the rings of a
kind and a few maps is good to a tenth, which every bound has on top.
"""

import numpy as np
import pytest
import torch

from s2fft_amd import _lib

pytestmark = pytest.mark.gpu


def _kind(n, back):
    if n & (n - 1) == 0:
        if n < 64:
            return "powers of two below 64", 2.8e-16 if back else 1.2e-16
        return ("powers of two to 256", 2.6e-16) if n <= 256 else \
            ("powers of two to 1024", 3.5e-16) if n <= 1024 else ("powers of two", 4.5e-16)
    if n < 64:
        return ("short", 4.9e-16) if n in (12, 20, 28, 44, 52) else (None, 0.0)
    return ("to 400", 6.6e-16) if n <= 400 else ("to 1100", 7.3e-16) if n <= 1100 else \
        ("long", 8.3e-16)


def _error2(got, want):
    return float((abs(got - want) ** 2).sum() / (abs(want) ** 2).sum())


@pytest.mark.parametrize("nside,L,batch", [(100, 211, 4), (256, 512, 2), (512, 1024, 1)])
def test_rms_error(nside, L, batch):
    rng = np.random.default_rng(nside)
    f = rng.standard_normal((batch, 12 * nside**2)) + 1j * rng.standard_normal(
        (batch, 12 * nside**2))
    spec = rng.standard_normal((batch, 4 * nside - 1, 2 * L)) + 1j * rng.standard_normal(
        (batch, 4 * nside - 1, 2 * L))
    lib, stream = _lib.lib(), torch.cuda.current_stream().cuda_stream
    ft, st = torch.from_numpy(f).cuda(), torch.from_numpy(spec).cuda()
    out, back = torch.empty_like(st), torch.empty_like(ft)
    _lib.check(lib.s2h_healpix_fft_prepare(nside, L))
    _lib.check(lib.s2h_healpix_fft(nside, L, 0, ft.data_ptr(), out.data_ptr(), batch, stream))
    _lib.check(lib.s2h_healpix_ifft(nside, L, 0, st.data_ptr(), back.data_ptr(), batch, stream))
    out, back = out.cpu().numpy(), back.cpu().numpy()
    m, at, seen = np.arange(-L, L), 0, {}
    for r in range(4 * nside - 1):
        n = 4 * min(r + 1, 4 * nside - 1 - r, nside)
        for b in range(batch):
            want = np.fft.fft(f[b, at:at + n].astype(np.clongdouble))[m % n]
            seen.setdefault(_kind(n, False) + (False,), []).append(_error2(out[b, r], want))
            fold = np.zeros(n, np.clongdouble)
            np.add.at(fold, m % n, spec[b, r].astype(np.clongdouble))
            seen.setdefault(_kind(n, True) + (True,), []).append(
                _error2(back[b, at:at + n], np.fft.ifft(fold) * n))
        at += n
    for (kind, bound, direction), e2 in seen.items():
        assert kind is None or np.sqrt(np.mean(e2)) < 1.1 * bound, (kind, direction)
