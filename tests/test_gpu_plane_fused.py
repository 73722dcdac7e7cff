"""Grids whose y and z passes run in one launch per RK stage, a block per
x-plane: the smallest and largest in each precision, with and without a
column count above 2 (n/2+1), single and in a batch, against the oracle (FP64,
1e-12, the bar of the other step tests) and against the FP64 state (mixed:
the increments of 3 steps carry float's 2^-24 times the transforms' growth of
about 30, 2e-6 of the largest coefficient)."""
import numpy as np
import pytest

import dns_amd
from conftest import random_field, rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8, 12, 18, 32, 48, 54, 64, 72])
def test_steps_match_oracle_and_mixed(oracle, n):
    print(f"plane pass n={n}", flush=True)
    u, nu, dt = random_field(n, seed=3 * n), 0.02, 0.1 / n
    o = oracle.solver(n, nu, dt)
    o.load_velocity(u)
    o.step(3)
    want, stale = o.get_spectral(), o.get_stale_velocity()
    o.close()
    for precision, tol in (("fp64", 1e-12), ("mixed", 2e-6), ("mixed_acc64", 2e-6)):
        with dns_amd.Batch([n, n], nu, [dt, dt / 2], precision) as b, dns_amd.Solver(n, nu, dt, precision) as s:
            s.load_velocity(u)
            b.load_velocity(0, u)
            b.load_velocity(1, u)
            s.step(3)
            b.step(3)
            got = s.get_spectral()
            assert rel(got, want) < tol and rel(s.get_stale_velocity(), stale) < 10 * tol, precision
            assert np.array_equal(b.get_spectral(0), got), precision
            assert not np.array_equal(b.get_spectral(1), got), precision
