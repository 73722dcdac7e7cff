"""Host logic of the offline radix tuner (dns_amd/tune_radix.py): the table
it reads back and the candidate schedules it would build (no GPU)."""
import math
import os
import re

import pytest

from dns_amd import build, roofline, tune_radix


def ends_divide(e, rad):
    return e % rad[0] == 0 and e % rad[-1] == 0


def test_table_covers_every_grid_size():
    for precision in ("fp64", "mixed"):
        t = tune_radix.table(precision)
        assert sorted(t) == sorted(build.grid_sizes())
        for n, (e, rad) in t.items():
            assert math.prod(rad) == n, (n, rad)
            assert ends_divide(e, rad) and set(rad) <= set(tune_radix.RADICES), (n, e, rad)
            assert n % e == 0 and (precision == "mixed" or roofline.elements_per_thread(n) == e)
    assert tune_radix.table("mixed")[64] == (8, (8, 8)) and tune_radix.table()[64] == (4, (4, 4, 4))


def test_the_table_is_the_only_one_and_every_radix_has_a_butterfly():
    """A candidate is compared with the schedule that the library runs: one
    row a size, or one of each precision, and none that no kernel reaches; the
    tuner's radices are those that the kernels implement."""
    with open(os.path.join(build.CSRC, "fft_engine.hpp")) as f:
        src = f.read()
    rows = re.findall(r"^(DNS_SCHED\w*)\((\d+),", src, re.M)
    assert {m for m, _ in rows} == {"DNS_SCHED", "DNS_SCHED_FLOAT"} and len(set(rows)) == len(rows)
    assert sorted(int(n) for m, n in rows if m == "DNS_SCHED") == sorted(build.grid_sizes())
    assert "struct Sched : std::conditional_t<sizeof(R) == 4, SchedFloat<N>, SchedTable<N>> {};" in src
    assert sorted(tune_radix.RADICES) == sorted({int(r) for r in re.findall(r"RAD == (\d+)", src)})


def test_candidates_are_the_fewest_stage_orderings():
    for n, precision in [(n, p) for n in build.grid_sizes() for p in ("fp64", "mixed")]:
        t = tune_radix.table(precision)
        e, cands = tune_radix.candidates(n, precision)
        assert e == t[n][0]
        assert cands[0] == t[n][1]                      # the table's own schedule first
        assert len(set(cands)) == len(cands)
        stages = {len(c) for c in cands[1:]}            # one stage count: the fewest
        assert len(stages) <= 1 and all(s <= len(t[n][1]) for s in stages), (n, stages)
        for c in cands:
            assert math.prod(c) == n and ends_divide(e, c)
    # counts that follow from the radix multisets (n = 2^a 3^b)
    assert len(tune_radix.candidates(486)[1]) == 1      # 9-6-9 only
    assert set(tune_radix.candidates(96)[1]) == {(4, 6, 4), (4, 12, 2), (2, 12, 4)}
    assert set(tune_radix.candidates(512)[1]) == {(8, 8, 8), (8, 16, 4), (4, 16, 8)}
    assert tune_radix.candidates(1024)[1] == [(8, 8, 4, 4), (8, 16, 8)]


def test_candidate_library_names_are_distinct():
    for n in (64, 128):
        assert len({tune_radix.name(n, e, c) for e, c in tune_radix.builds(n)}) == len(tune_radix.builds(n))
    assert set(tune_radix.builds(64)) >= {(4, (4, 4, 4)), (8, (8, 8))}


@pytest.mark.parametrize("e,rad", tune_radix.builds(64))
def test_every_candidate_of_a_size_with_two_schedules_compiles(e, rad):
    """A candidate build replaces the schedules of both precisions."""
    flags = ["-DDNS_N=64", "-DDNS_SCHED_N=64", f"-DDNS_SCHED_E={e}", "-DDNS_SCHED_R=" + ",".join(map(str, rad))]
    build._run([build.HIPCC, *build.HIP_FLAGS, *flags, "-fsyntax-only", os.path.join(build.CSRC, "inst.hip")])
