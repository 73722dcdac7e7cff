"""Transforms of the schedules with radices 6, 9, 12 and 16 and partly filled
middle stages, against numpy: forward, inverse and round trip in both
precisions, on fields with content at every wavenumber including Nyquist.

Tolerance: each of the at most four stages per axis multiplies the 2-norm of
the rounding error by less than 1 + 8 u (a radix-16 butterfly sums 16 terms in
four levels, twiddles add one rounding), so three axes stay below 100 u
relative to the 2-norm; u = 2^-53 or 2^-24."""
import numpy as np
import pytest

import dns_amd

pytestmark = pytest.mark.gpu


# one of each radix and of each way a middle stage or a z block is filled:
# radix 6 alone (36), a middle 3 or 6 on 4-element threads (48, 96), z blocks
# of several pencils (144, 288), an odd count of elements with a middle 16 or
# 6 (432, 486); the size tests step every grid
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("n", [12, 24, 36, 48, 96, 144, 162, 288, 432, 486])
def test_transforms_match_numpy(n, precision):
    print(f"wide radices n={n} {precision}", flush=True)
    u = 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    a = np.random.default_rng(n).standard_normal((n, n, n))
    with dns_amd.Solver(n, 0.01, 0.01, precision) as s:
        f = s.rfft3(a)
        b = s.irfft3(f) / float(n) ** 3
    want = np.fft.rfftn(a)
    assert np.linalg.norm(f - want) <= 100 * u * np.linalg.norm(want)
    assert np.linalg.norm(b - a) <= 200 * u * np.linalg.norm(a)
