"""FP64 transforms against long double: the error stays that of the schedules of
radices 4, 3 and 2 that these grids had before, measured on the same inputs (2-norm,
forward and inverse).  Radix-6 butterflies and another order of the radices had
raised it by up to 9% through the rounding of their constants, which is alike in
every butterfly and axis.  2% for the sampling of the smallest grid's
few coefficients and for orders of the radices whose constants cancel less."""
import numpy as np
import pytest

import dns_amd

pytestmark = pytest.mark.gpu

FORMER = {12: (2.079e-16, 2.251e-16), 24: (2.265e-16, 2.280e-16), 48: (2.503e-16, 2.482e-16),
          72: (2.915e-16, 2.895e-16), 96: (2.738e-16, 2.687e-16), 128: (3.072e-16, 3.005e-16),
          144: (3.034e-16, 2.982e-16), 192: (2.980e-16, 2.886e-16), 216: (3.581e-16, 3.543e-16)}


@pytest.mark.parametrize("n", sorted(FORMER))
def test_transform_error_is_no_larger_than_before(n):
    print(f"transform error n={n}", flush=True)
    a = np.random.default_rng(n).standard_normal((n, n, n))
    want = np.fft.rfftn(a.astype(np.longdouble))
    spec = want.astype(np.complex128)
    back = np.fft.irfftn(spec.astype(np.clongdouble), s=(n, n, n), axes=(0, 1, 2)) * np.longdouble(n) ** 3
    with dns_amd.Solver(n, 0.01, 0.01) as s:
        f, b = s.rfft3(a), s.irfft3(spec)
    forward = np.sqrt(np.sum(np.abs(f - want) ** 2) / np.sum(np.abs(want) ** 2))
    inverse = np.sqrt(np.sum((b - back) ** 2) / np.sum(back ** 2))
    print(f"  forward {forward:.3e} inverse {inverse:.3e}", flush=True)
    assert forward <= 1.02 * FORMER[n][0] and inverse <= 1.02 * FORMER[n][1]
