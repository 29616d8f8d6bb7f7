"""The schedule tuner times schedules on the units that the full input will have,
tries a unit size once, and knows the merge's default work item (CPU, with a
context that only records what it is asked)."""
from types import SimpleNamespace

import numpy as np
import pytest

from ggcat_amd.autotune import Schedule, autotune, default_grid, load_grid, sample_fraction, unit_size
from ggcat_amd.native import HASH_SEQ, Params


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
        n_sub = ((1 << params.buckets_log) + 1) << params.second_buckets_log
        self.unit = unit_size(n_bytes, n_sub, self.knobs["unit_bytes"])
        self.runs.append((dict(self.knobs), self.unit))

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


@pytest.mark.parametrize("k,ratio", [(31, 16), (63, 16), (31, 15), (63, 11)])
def test_schedules_run_on_the_full_units(k, ratio):
    p = Params(k, 15, 3, 1, 0, HASH_SEQ, 2)  # 18 sub-buckets
    n_sub, full = 18, 18 * 61_200
    ctx = _Recorder()
    out = autotune(ctx, np.zeros(full // ratio, np.uint8), p, repeats=1, full_bytes=full)
    assert out["tried"] == len(ctx.runs) > 5
    want = {unit_size(full, n_sub, s.unit_bytes) for s in default_grid(k)}
    got = {unit for _, unit in ctx.runs}
    for u in got:  # within a factor of sqrt(2), and the same where the sample is a power of two smaller
        near = min(want, key=lambda w: abs(np.log(u / w)))
        assert abs(u - near) <= 1 if ratio == 16 else abs(np.log2(u / near)) <= 0.51
    # a unit size that several values of unit_bytes come to is tried once
    first = [(tuple(sorted((a, b) for a, b in kn.items() if a != "unit_bytes")), unit) for kn, unit in ctx.runs]
    assert len(set(first)) == len(first)
    assert out["schedule"]["unit_bytes"] in {s.unit_bytes for s in default_grid(k)}


def test_best_schedule_is_the_one_of_the_full_units():
    """A table of 1024 entries is fast with units of 1000 bytes and slow with the 1900 of the full input."""
    p = Params(31, 15, 3, 1, 0, HASH_SEQ, 2)
    full = 18 * 1913 * 32
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
