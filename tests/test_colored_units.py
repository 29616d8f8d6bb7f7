"""Default unit size of colored builds: where the merge's tables are smaller than
2048 entries (two-word keys, or more than 64 colors), units are small enough for
most work items to fit a table.  Twice as large ones split several times as many
items, each of which reads its records once per part."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_RK128, HASH_SEQ, GpuContext, Params


def _splits(ctx, data, starts, colors, k, m, kind, b, sb, unit_bytes):
    ctx.set_tuning(unit_bytes=unit_bytes, merge_wgs_per_cu=1)
    try:
        ctx.bucketing(data, Params(k, m, b, sb, 0, kind, 1), colors=(starts, colors))
        ctx.kmers_merge()
        return int(ctx.counters()[4])
    finally:
        ctx.set_tuning()


def _check(ctx, scale, n, k, m, kind, b, sb):
    gs = synth.config3_genomes(scale, n)
    data, starts = synth.contigs_joined(gs, 5, 3000, 9000)
    colors = np.arange(n, dtype=np.uint32)
    by_default = _splits(ctx, data, starts, colors, k, m, kind, b, sb, 0)
    large = _splits(ctx, data, starts, colors, k, m, kind, b, sb, 2000)
    assert large >= 4 and 2 * by_default < large, (by_default, large)


def test_colored_units_emulated():
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    # 20 KB over 3 sub-buckets: 4 units of 1650 bytes in each, or 8 of 825
    _check(ctx, 0.0004, 16, 45, 21, HASH_SEQ, 1, 0)
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("scale,n,k,m,kind", [(0.2, 16, 45, 21, HASH_SEQ), (0.2, 16, 63, 21, HASH_RK128), (0.1, 96, 31, 15, HASH_SEQ)])
def test_colored_units(gpu_ctx, scale, n, k, m, kind):
    print(f"case colored units n={n} k={k} kind={kind}", flush=True)
    _check(gpu_ctx, scale, n, k, m, kind, 8, 2)
