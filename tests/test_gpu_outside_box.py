"""Modes outside the dealiased box only diffuse: their stage state and
accumulator are formed from the step's first state instead of being stored,
so the RK4 polynomial of z = nu dt |k|^2 has to come out mode by mode, while
the modes inside follow the oracle (FP64).

Tolerances: a step does at most 16 roundings on a mode, each of relative size
u = 2^-53 of values no larger than (1 + z)^3 |U|; in the mixed forms the
increments, of size at most z (1 + z)^3 |U|, carry 2^-24 instead."""
import numpy as np
import pytest

import dns_amd
from conftest import random_field, rel, rk4_amplification, wavenumbers

pytestmark = pytest.mark.gpu


# smallest grids, a box edge between two rows of a pair (n=18: nk = 7), one on
# it (n=64: kmax = 22 exactly), pencils of threes, a tile cut by the box edge
@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed_acc64"])
@pytest.mark.parametrize("n", [8, 12, 18, 54, 64, 128])
def test_modes_outside_the_box_diffuse(oracle, n, precision):
    print(f"outside the box n={n} {precision}", flush=True)
    nu, dt, steps = 0.02, 0.2 / n, 3
    with dns_amd.Solver(n, nu, dt, precision) as s:
        u = random_field(n, seed=n)
        s.load_velocity(u)
        a = s.get_spectral()
        s.step(steps)
        b = s.get_spectral()
    kx, ky, kz = wavenumbers(n)
    kmax = 2.0 / 3.0 * (n // 2 + 1)
    outside = (np.abs(kx) >= kmax) | (np.abs(ky) >= kmax) | (np.abs(kz) >= kmax)
    z = np.broadcast_to(nu * dt * (kx * kx + ky * ky + kz * kz), outside.shape)[outside]
    want = a[:, outside] * rk4_amplification(z) ** steps
    tol = steps * 16 * (1 + z) ** 3 * 2.0 ** -53
    if precision != "fp64":
        tol = tol + steps * 16 * z * (1 + z) ** 3 * 2.0 ** -24
    # the amplification is of order one in every step (z below its stability
    # bound), so relative errors of the steps add up
    assert z.max() < 2.5
    scale = np.abs(a[:, outside])
    assert np.all(np.abs(b[:, outside] - want) <= tol * np.maximum(scale, np.abs(want)))
    if precision == "fp64" and n <= 64:
        o = oracle.solver(n, nu, dt)
        o.load_velocity(u)
        o.step(steps)
        assert rel(b, o.get_spectral()) < 1e-12
        o.close()
