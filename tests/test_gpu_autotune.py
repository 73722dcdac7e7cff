"""dns_autotune times every launch shape that differs from the lower ones, once:
counted through the kernel timing, which brackets the launches of its steps.
All four shapes stay selectable."""
import pytest

import dns_amd
from conftest import random_field

pytestmark = pytest.mark.gpu


# y and z passes in one launch per plane, so no z block to widen (FP64 up to 48,
# mixed up to 72); pencils of 18 threads, whose second set would cross a wave
# (108); both bits (64 FP64)
@pytest.mark.parametrize("n,precision,shapes", [(16, "fp64", 2), (48, "mixed", 2), (72, "mixed", 2), (108, "fp64", 2),
                                                (64, "fp64", 4)])
def test_autotune_times_each_launch_once(n, precision, shapes):
    print(f"autotune n={n} {precision}", flush=True)
    steps = 2
    with dns_amd.Solver(n, 0.01, 0.1 / n, precision) as s:
        s.load_velocity(random_field(n, n))
        assert s.launch_shapes() == 4
        for shape in range(4):
            s.set_launch_shape(shape)
            s.step(1)
        s.set_kernel_timing(True)
        best = s.autotune(steps)
        assert 0 <= best < 4 and best == s.launch_shape() and (shapes == 4 or best < 2)
        assert s.kernel_timing()["zfused.s1"][1] == shapes * (steps + 1)
