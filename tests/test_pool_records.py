"""Records longer than a slot (the long-record pool) through every staging block
size and every merge variant: records and solid tables against the oracle, on
the CPU emulation.  The inputs hold long runs whose windows all have the same
minimum, so groups that start far before their tile are among them."""
import numpy as np
import pytest

from ggcat_amd.native import HASH_RK128, HASH_SEQ, GpuContext, Params
from oracle import binding as O
from tests.helpers import (adversarial_records, bitmaps_from_sets, colored_solid_array, inline_capacity, joined,
                           record_tuples, solid_array)

# window widths 2 to 50 (blocks 2, 4, 8, 16), slots of 4, 8 and 16 words, one- and two-word keys, both hashes
CASES = [(9, 7, HASH_SEQ, 0), (15, 8, HASH_SEQ, 0), (24, 12, HASH_SEQ, 0), (32, 12, HASH_SEQ, 0), (32, 25, HASH_RK128, 0),
         (12, 6, HASH_RK128, 0), (33, 31, HASH_SEQ, 0), (47, 14, HASH_SEQ, 0), (46, 35, HASH_RK128, 0),
         (64, 21, HASH_SEQ, 0), (64, 14, HASH_RK128, 0), (31, 10, HASH_SEQ, 3), (31, 23, HASH_SEQ, 70),
         (45, 21, HASH_SEQ, 3), (63, 21, HASH_RK128, 3)]


def _records(k: int) -> list[bytes]:
    recs = adversarial_records(np.random.default_rng(700 + k))
    # two copies of the runs and repeats, so that equal pool records meet
    return recs[:16] + [r[:2300] for r in recs[16:19]] + recs[9:14] + recs[19:27]


@pytest.fixture(scope="module")
def emu_ctx():
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    ctx.set_tuning(merge_wgs_per_cu=1)
    yield ctx
    ctx.close()


@pytest.mark.parametrize("k,m,kind,colors", CASES)
def test_pool_records_emulated(emu_ctx, k, m, kind, colors):
    recs = _records(k)
    data = joined(recs)
    b, sb = 3, 1
    p = Params(k, m, b, sb, 0, kind, 1)
    if not colors:
        emu_ctx.bucketing(data, p)
        o = O.bucketing(data, k, m, b, sb, threads=2)
    else:
        at = np.cumsum([len(r) + 1 for r in recs])
        starts = np.array([0, at[6], at[20]], np.uint64)
        ids = np.array([colors - 1, 0, 1], np.uint32)
        emu_ctx.bucketing(data, p, colors=(starts, ids))
        o = O.bucketing_colored(data, k, m, b, sb, starts, ids, threads=2)
    r = o.records()
    assert int(r["length"].max()) > inline_capacity(k, m)
    assert record_tuples(emu_ctx.records()) == record_tuples(r)
    emu_ctx.kmers_merge()
    o.merge(k, b, sb, kind, 1, 2)
    if not colors:
        assert np.array_equal(solid_array(emu_ctx.solid()), solid_array(o.solid()))
    else:
        off, cols = o.solid_colors()
        want = colored_solid_array(o.solid(), bitmaps_from_sets(off, cols, (colors + 31) // 32))
        assert np.array_equal(colored_solid_array(emu_ctx.solid(), emu_ctx.solid_colors()), want)


def test_rolled_records_emulated(emu_ctx):
    # no_dedup = 2 names a mode of the seq hash; rabin-karp128 gives the same table with and without it
    data = joined(_records(46)[:14])
    emu_ctx.set_tuning(merge_wgs_per_cu=1, no_dedup=2)
    try:
        for k, m, kind in ((31, 15, HASH_SEQ), (45, 21, HASH_SEQ), (45, 21, HASH_RK128)):
            emu_ctx.bucketing(data, Params(k, m, 2, 1, 0, kind, 1))
            emu_ctx.kmers_merge()
            o = O.bucketing(data, k, m, 2, 1, threads=2)
            o.merge(k, 2, 1, kind, 1, 2)
            assert np.array_equal(solid_array(emu_ctx.solid()), solid_array(o.solid()))
    finally:
        emu_ctx.set_tuning(merge_wgs_per_cu=1)
