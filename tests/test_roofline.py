"""Byte counts of dns_amd/roofline.py (no GPU): the modes that the x pass
stores and reads, and the thresholds it shares with the kernels' sources."""
import os
import re

import numpy as np
import pytest

from conftest import wavenumbers
from dns_amd import build, roofline


def _source(name):
    with open(os.path.join(build.CSRC, name)) as f:
        return f.read()


def test_thresholds_are_the_kernels():
    first, = re.findall(r"constexpr bool SKIP = N >= (\d+);", _source("kernels.hpp"))
    d, f = re.findall(r"constexpr bool PLANE = N <= \(sizeof\(R\) == 8 \? (\d+) : (\d+)\)", _source("engine.hpp"))[0]
    for n in build.grid_sizes():
        assert roofline.stores_all_modes(n) == (n < int(first))
        assert roofline.plane_fused(n, "fp64") == (n <= int(d))
        assert roofline.plane_fused(n, "mixed") == (n <= int(f))


# both sides of the first grid that leaves the outer modes unstored
@pytest.mark.parametrize("n", [16, 64, 72, 96, 108])
def test_x_pass_bytes_by_mode_count(n):
    """E's bytes from a count of the modes: the nonlinear term in the rows of
    the box, and per mode what each stage reads and writes of Un, Ur and the
    accumulator (16 bytes a value in FP64; float copy of Un, Ur and S in mixed)."""
    kx, ky, kz = wavenumbers(n)
    kmax = 2.0 / 3.0 * (n // 2 + 1)
    inside = (np.abs(kx) < kmax) & (np.abs(ky) < kmax) & (kz < kmax)
    rows = n * int(np.sum((np.abs(ky) < kmax) & (kz < kmax)))
    every = inside.size
    kept = every if n < 96 else int(np.sum(inside))
    fp64 = {1: every + 2 * kept, 2: every + 4 * kept, 3: every + 4 * kept, 4: kept + 2 * every}
    mixed = {1: every + 2 * kept, 2: every + 4 * kept, 3: every + 4 * kept, 4: 2 * kept + 5 * every}
    for precision, size, modes in (("fp64", 16, fp64), ("mixed", 8, mixed)):
        b = roofline.slot_bytes(n, precision)
        for stage, m in modes.items():
            assert b[f"xfwd_rk.s{stage}"] == 3 * size * (rows + m), (precision, stage)
