"""Boundary k-mers counted half in each of two work items whose color sets span
1, 3 and 32 words: their halves combined on the device, against the oracle, with
fewer entries than a wavefront compares at a time and with more."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_SEQ, GpuContext, Params
from oracle import binding as O
from tests.helpers import bitmaps_from_sets, colored_solid_array


def _check(ctx, k, m, scale, n, top, lo, hi):
    gs = synth.config3_genomes(scale, n)
    data, starts = synth.contigs_joined(gs, 5, 3000, 9000)
    colors = (np.arange(n, dtype=np.uint32) * 29) % top
    colors[0] = top - 1
    ctx.set_tuning(unit_bytes=100, item_occ=64, merge_wgs_per_cu=2)
    try:
        ctx.bucketing(data, Params(k, m, 1, 1, 0, HASH_SEQ, 1), colors=(starts, colors))
        ctx.kmers_merge()
        assert lo <= int(ctx.counters()[6]) <= hi, int(ctx.counters()[6])
        o = O.bucketing_colored(data, k, m, 1, 1, starts, colors, threads=4)
        o.merge(k, 1, 1, HASH_SEQ, 1, 4)
        off, cols = o.solid_colors()
        want = colored_solid_array(o.solid(), bitmaps_from_sets(off, cols, (top + 31) // 32))
        assert np.array_equal(colored_solid_array(ctx.solid(), ctx.solid_colors()), want)
    finally:
        ctx.set_tuning()


@pytest.mark.parametrize("k,m,top", [(31, 15, 1024), (45, 21, 70)])
def test_fixup_colors_emulated(k, m, top):
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    _check(ctx, k, m, 0.0002, 4, top, 2, 4096)
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("k,m,scale,n,top,lo,hi", [(31, 15, 0.0002, 4, 1024, 2, 400), (31, 15, 0.002, 12, 1024, 500, 4096),
                                                   (45, 21, 0.002, 12, 70, 500, 4096), (31, 15, 0.002, 12, 30, 500, 4096),
                                                   (31, 15, 0.02, 40, 1024, 4097, 1 << 30)])
def test_fixup_colors(gpu_ctx, k, m, scale, n, top, lo, hi):
    print(f"case fixup colors k={k} n={n} top={top}", flush=True)
    _check(gpu_ctx, k, m, scale, n, top, lo, hi)
