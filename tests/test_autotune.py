"""The schedule tuner times schedules on the units and sub-buckets that the full
input will have, tries a unit size once, and knows the merge's default work item (CPU, with a
context that only records what it is asked)."""
from types import SimpleNamespace

import numpy as np
import pytest

from ggcat_amd.autotune import (Schedule, autotune, default_grid, load_grid, n_sub, sample_fraction, sample_params, unit_log,
                                unit_size)
from ggcat_amd.native import HASH_SEQ, Params

N_SUB = 9 << 5  # sub-buckets of buckets_log 3, second_buckets_log 5


class _Recorder:
    """Timings come from `cost(knobs, unit size)`, in ms."""

    def __init__(self, cost=lambda knobs, unit: 1.0):
        self.cost, self.knobs, self.runs = cost, {}, []

    def set_tuning(self, **kw):
        self.knobs = kw

    def upload(self, a):
        return 1, a.size

    def free(self, ptr):
        pass

    def bucketing(self, data, params, device_ptr=None, n_bytes=None):
        self.unit = unit_size(n_bytes, n_sub(params), self.knobs["unit_bytes"])
        self.runs.append((dict(self.knobs), self.unit, unit_log(n_bytes, n_sub(params), self.knobs["unit_bytes"])))

    def kmers_merge(self):
        pass

    def timings(self):
        t = np.zeros(9)
        t[6] = self.cost(self.knobs, self.unit)
        return t

    def solid(self):
        z = np.zeros(0, np.uint32)
        return SimpleNamespace(keys=np.zeros((0, 1), np.uint64), sub=z, mult=z, flags=z)


def test_unit_size():
    # 4.016 GB over 65600 sub-buckets: the sizes the library halves down to
    assert [unit_size(4_016_000_000, 65600, u) for u in (1000, 2000, 3000)] == [956, 1913, 1913]
    assert [unit_size(268_435_213, 65600, u) for u in (1000, 2000, 3000)] == [511, 1023, 2046]
    assert unit_size(1000, 65600, 2000) == 0
    assert unit_size(4_016_000_000, 65600, 1) == 4_016_000_000 // 65600 // 256  # 2^25 units at most
    assert unit_size(1 << 30, 18, 1) == (1 << 20) // 18  # 10 halvings at most


@pytest.mark.parametrize("full", [4_016_000_000, 15_100_000_000, 250_000_000, 1 << 28])
def test_sample_units_are_the_full_ones(full):
    f = sample_fraction(full, 256 << 20)
    n = round(full * f)
    assert n <= 256 << 20 and (full <= 256 << 20 or 2 * n > 256 << 20)
    for u in (1400, 2000, 3000):
        a, b = unit_size(full, 65600, u), unit_size(n, 65600, u)
        assert abs(a - b) <= 1


@pytest.mark.parametrize("full,sample,b,sb,want", [(1 << 32, 1 << 28, 10, 6, (10, 2)), (1 << 32, 1 << 22, 10, 6, (6, 0)),
                                                   (1 << 32, 3 << 26, 10, 6, (10, 2)), (1 << 20, 1 << 20, 4, 2, (4, 2)),
                                                   (1000, 1 << 20, 4, 2, (4, 2)), (1 << 32, 1 << 20, 3, 1, (1, 0))])
def test_sample_sub_buckets(full, sample, b, sb, want):
    q = sample_params(Params(31, 15, b, sb, 0, HASH_SEQ, 2), full, sample)
    assert (q.buckets_log, q.second_buckets_log) == want and (q.k, q.m, q.hash_kind, q.min_multiplicity) == (31, 15, HASH_SEQ, 2)


@pytest.mark.parametrize("k,ratio", [(31, 16), (63, 16), (31, 15), (63, 11)])
def test_schedules_run_on_the_full_units(k, ratio):
    p = Params(k, 15, 3, 5, 0, HASH_SEQ, 2)
    full = N_SUB * 61_200
    ctx = _Recorder()
    out = autotune(ctx, np.zeros(full // ratio, np.uint8), p, repeats=1, full_bytes=full)
    assert out["tried"] == len(ctx.runs) > 5
    want = {unit_size(full, N_SUB, s.unit_bytes) for s in default_grid(k)}
    for _, unit, log in ctx.runs:
        near = min(want, key=lambda w: abs(np.log(unit / w)))
        # where the sample is smaller by a power of two both are those of the full input
        assert abs(unit - near) <= 1 if ratio == 16 else abs(np.log2(unit / near)) <= 0.51
        if ratio == 16:
            assert log in {unit_log(full, N_SUB, s.unit_bytes) for s in default_grid(k)}
    # a unit size that several values of unit_bytes come to is tried once
    first = [(tuple(sorted((a, b) for a, b in kn.items() if a != "unit_bytes")), unit) for kn, unit, _ in ctx.runs]
    assert len(set(first)) == len(first)
    assert out["schedule"]["unit_bytes"] in {s.unit_bytes for s in default_grid(k)}


def test_best_schedule_is_the_one_of_the_full_units():
    """A table of 1024 entries is fast with units of 1000 bytes and slow with the 1900 of the full input."""
    p = Params(31, 15, 3, 5, 0, HASH_SEQ, 2)
    full = N_SUB * 1913 * 32
    ctx = _Recorder(lambda kn, unit: 1.0 if kn["lds_table_log"] != 10 else 0.5 if unit < 1200 else 2.0)
    out = autotune(ctx, np.zeros(full // 15, np.uint8), p, repeats=1, full_bytes=full)
    assert out["schedule"]["lds_table_log"] != 10


def test_second_stage_skips_the_default_once():
    for k, log, default in ((31, 11, 1024), (31, 10, 512), (47, 10, 768), (63, 10, 768), (64, 10, 512)):
        lds = 1 << log
        got = [(s.table_pct, s.item_occ) for s in load_grid(Schedule(unit_bytes=2000, table_pct=200, lds_table_log=log), k)
               if not s.no_dedup]
        want = {(t, o) for t in (100, 200, 400) for o in (lds // 2, lds, 2 * lds)} - {(200, default)}
        assert set(got) == want and len(got) == len(want)
