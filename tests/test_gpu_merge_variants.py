"""Every merge variant (key width, hash, slot words, colors) at the ends of its
k range, with records placed by position and hashed, and with work items split
by the table's size, against the oracle."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_RK128, HASH_SEQ, GpuContext, Params
from oracle import binding as O
from tests.helpers import bitmaps_from_sets, colored_solid_array, solid_array

# k = 32 | 33 and 63 | 64 part the key widths; (31, 10), (32, 12) have 8-word slots, (33, 31) 4-word
# slots under two-word keys, (64, 14) 16-word slots
CASES = [(31, 15, HASH_SEQ), (31, 10, HASH_SEQ), (32, 12, HASH_SEQ), (32, 25, HASH_RK128), (12, 6, HASH_RK128),
         (33, 31, HASH_SEQ), (33, 14, HASH_SEQ), (46, 21, HASH_RK128), (47, 14, HASH_SEQ), (62, 21, HASH_RK128),
         (63, 21, HASH_SEQ), (63, 21, HASH_RK128), (64, 21, HASH_SEQ), (64, 20, HASH_RK128), (64, 14, HASH_SEQ)]


def _data(genome: int, k: int) -> np.ndarray:
    g = synth.genome(81 + k, genome, repeat_frac=0.2, rep_min=200, rep_max=400)
    return synth.reads(g, 82, genome // 8, 150, 0.01)


def _check(ctx, data, k, m, kind, s):
    ctx.bucketing(data, Params(k, m, 3, 2, 0, kind, s))
    ctx.kmers_merge()
    o = O.bucketing(data, k, m, 3, 2, threads=4)
    o.merge(k, 3, 2, kind, s, 4)
    got, want = solid_array(ctx.solid()), solid_array(o.solid())
    assert want.shape[0] > 0 and got.shape == want.shape and np.array_equal(got, want)


@pytest.fixture(scope="module")
def emu_ctx():
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    ctx.set_tuning(merge_wgs_per_cu=1)
    yield ctx
    ctx.close()


@pytest.mark.parametrize("k,m,kind", CASES)
def test_merge_variants_emulated(emu_ctx, k, m, kind):
    _check(emu_ctx, _data(1200, k), k, m, kind, 2)


@pytest.mark.gpu
@pytest.mark.parametrize("no_dedup", [0, 3])
@pytest.mark.parametrize("k,m,kind", CASES)
def test_merge_variants(gpu_ctx, k, m, kind, no_dedup):
    print(f"case merge variant k={k} m={m} kind={kind} no_dedup={no_dedup}", flush=True)
    # 60 kbp over 36 sub-buckets: items above one table, split by the size of
    # the table, and (4 MiB units) with records hashed
    gpu_ctx.set_tuning(no_dedup=no_dedup, unit_bytes=(1 << 22) if no_dedup else 0)
    try:
        _check(gpu_ctx, _data(60_000, k), k, m, kind, 1 if no_dedup else 2)
    finally:
        gpu_ctx.set_tuning()


@pytest.mark.gpu
@pytest.mark.parametrize("k,m,kind,n", [(31, 15, HASH_SEQ, 32), (32, 12, HASH_SEQ, 33), (33, 21, HASH_SEQ, 40),
                                        (63, 21, HASH_SEQ, 64), (64, 21, HASH_SEQ, 40), (45, 21, HASH_RK128, 40)])
def test_colored_merge_variants(gpu_ctx, k, m, kind, n):
    print(f"case colored merge variant k={k} m={m} kind={kind} colors={n}", flush=True)
    gs = synth.config3_genomes(0.004, n)
    data, starts = synth.contigs_joined(gs, 5, 3000, 9000)
    colors = np.arange(n, dtype=np.uint32)
    gpu_ctx.bucketing(data, Params(k, m, 4, 2, 0, kind, 1), colors=(starts, colors))
    gpu_ctx.kmers_merge()
    o = O.bucketing_colored(data, k, m, 4, 2, starts, colors, threads=4)
    o.merge(k, 4, 2, kind, 1, 4)
    off, cols = o.solid_colors()
    want = colored_solid_array(o.solid(), bitmaps_from_sets(off, cols, (n + 31) // 32))
    assert np.array_equal(colored_solid_array(gpu_ctx.solid(), gpu_ctx.solid_colors()), want)
