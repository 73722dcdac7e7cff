"""Modes outside the dealiased box only diffuse: from n=96 on their stage state
and accumulator are formed from the step's first state instead of being stored,
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


def _random_spectrum(n):
    """Coefficients of a velocity of order one with content at every
    wavenumber; the planes kz = 0 and n/2 are not symmetric, whose modes outside
    the box diffuse all the same."""
    kx, ky, kz = wavenumbers(n)
    a = np.random.default_rng(n).standard_normal((3, n, n, n // 2 + 1, 2)).view(np.complex128)[..., 0]
    a *= n ** 1.5 * np.exp(-(kx * kx + ky * ky + kz * kz) / (0.08 * n * n))
    return a


# the last grid that stores all modes with an integer kmax (64: 22) and the
# first that does not (96); 6 elements per thread (108, 162: half-filled
# middle stage); 16 float elements in the x pass (192); an integer kmax (256:
# 86) with the outer modes unstored; an odd element count (432: 9), where the
# epilogue takes one position at a time in double and three in float
@pytest.mark.parametrize("precision", ["fp64", "mixed", "mixed_acc64"])
@pytest.mark.parametrize("n", [18, 64, 96, 108, 162, 192, 256, 432])
def test_modes_outside_the_box_diffuse(oracle, n, precision):
    print(f"outside the box n={n} {precision}", flush=True)
    nu, dt, steps = 0.02, 0.2 / n, 3
    u = random_field(n, seed=n) if n <= 192 else None
    with dns_amd.Solver(n, nu, dt, precision) as s:
        if u is None:
            s.load_velocity(np.zeros((3, n, n, n)))
            s.set_spectral(_random_spectrum(n))
        else:
            s.load_velocity(u)
        a = s.get_spectral()
        s.step(steps)
        b = s.get_spectral()
    kx, ky, kz = wavenumbers(n)
    kmax = 2.0 / 3.0 * (n // 2 + 1)
    outside = (np.abs(kx) >= kmax) | (np.abs(ky) >= kmax) | (np.abs(kz) >= kmax)
    z = np.broadcast_to(nu * dt * (kx * kx + ky * ky + kz * kz), outside.shape)[outside]
    tol = steps * 16 * (1 + z) ** 3 * 2.0 ** -53
    if precision != "fp64":
        tol = tol + steps * 16 * z * (1 + z) ** 3 * 2.0 ** -24
    # the amplification is of order one in every step (z below its stability
    # bound), so relative errors of the steps add up
    assert z.max() < 2.5
    amp = rk4_amplification(z) ** steps
    for f in range(3):
        a0 = a[f][outside]
        want = a0 * amp
        assert np.all(np.abs(b[f][outside] - want) <= tol * np.maximum(np.abs(a0), np.abs(want))), f
    if precision == "fp64" and u is not None:
        o = oracle.solver(n, nu, dt)
        o.load_velocity(u)
        o.step(steps)
        assert rel(b, o.get_spectral()) < 1e-12
        o.close()
