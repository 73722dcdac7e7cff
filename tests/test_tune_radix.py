"""Host logic of the offline radix tuner (dns_amd/tune_radix.py): the table
it reads back and the candidate schedules it would build (no GPU)."""
import math
import os
import re

from dns_amd import build, roofline, tune_radix


def ends_divide(e, rad):
    return e % rad[0] == 0 and e % rad[-1] == 0


def test_table_covers_every_grid_size():
    t = tune_radix.table()
    assert sorted(t) == sorted(build.grid_sizes())
    for n, (e, rad) in t.items():
        assert math.prod(rad) == n, (n, rad)
        assert ends_divide(e, rad) and set(rad) <= set(tune_radix.RADICES), (n, e, rad)
        assert n % e == 0 and roofline.elements_per_thread(n) == e


def test_the_table_is_the_only_one_and_every_radix_has_a_butterfly():
    """A candidate is compared with the schedule that the library runs: one
    row a size, no second table in front of it; the tuner's radices are those
    that the kernels implement."""
    with open(os.path.join(build.CSRC, "fft_engine.hpp")) as f:
        src = f.read()
    rows = re.findall(r"^DNS_SCHED\w*\((\d+),", src, re.M)
    assert sorted(map(int, rows)) == sorted(build.grid_sizes())
    assert "template <int N> struct Sched : SchedTable<N> {};" in src
    assert sorted(tune_radix.RADICES) == sorted({int(r) for r in re.findall(r"RAD == (\d+)", src)})


def test_candidates_are_the_fewest_stage_orderings():
    t = tune_radix.table()
    for n in sorted(t):
        e, cands = tune_radix.candidates(n)
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
    e, cands = tune_radix.candidates(128)
    names = {tune_radix.name(128, c) for c in cands}
    assert len(names) == len(cands)
