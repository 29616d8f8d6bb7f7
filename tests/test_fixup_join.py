"""Boundary k-mers counted half in each of two work items: their halves combined
on the device (a few thousand entries and fewer) and on the host (more), with
64- and 128-bit keys and with colors, against the oracle."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_RK128, HASH_SEQ, GpuContext, Params
from oracle import binding as O
from tests.helpers import bitmaps_from_sets, colored_solid_array, solid_array


def _check(ctx, k, m, kind, genome, lo, hi):
    """Units of a few hundred bytes: neighbouring groups of a sub-bucket mostly
    lie in different units."""
    data = synth.reads(synth.genome(81, genome), 82, genome // 10, 150, 0.005)
    ctx.set_tuning(unit_bytes=100, item_occ=64, merge_wgs_per_cu=2)
    try:
        ctx.bucketing(data, Params(k, m, 1, 1, 0, kind, 1))
        ctx.kmers_merge()
        assert lo <= int(ctx.counters()[6]) <= hi, int(ctx.counters()[6])
        o = O.bucketing(data, k, m, 1, 1, threads=4)
        o.merge(k, 1, 1, kind, 1, 4)
        assert np.array_equal(solid_array(ctx.solid()), solid_array(o.solid()))
    finally:
        ctx.set_tuning()


def _check_colored(ctx, scale):
    gs = synth.config3_genomes(scale, 12)
    data, starts = synth.contigs_joined(gs, 5, 3000, 9000)
    colors = (np.arange(12, dtype=np.uint32) * 29) % 60
    ctx.set_tuning(unit_bytes=100, item_occ=64, merge_wgs_per_cu=2)
    try:
        ctx.bucketing(data, Params(31, 15, 1, 1, 0, HASH_SEQ, 1), colors=(starts, colors))
        ctx.kmers_merge()
        assert 0 < int(ctx.counters()[6]) <= 4096, int(ctx.counters()[6])
        o = O.bucketing_colored(data, 31, 15, 1, 1, starts, colors, threads=4)
        o.merge(31, 1, 1, HASH_SEQ, 1, 4)
        off, cols = o.solid_colors()
        want = colored_solid_array(o.solid(), bitmaps_from_sets(off, cols, 2))
        assert np.array_equal(colored_solid_array(ctx.solid(), ctx.solid_colors()), want)
    finally:
        ctx.set_tuning()


@pytest.fixture(scope="module")
def emu_ctx():
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    yield ctx
    ctx.close()


@pytest.mark.parametrize("k,m,kind", [(31, 15, HASH_SEQ), (45, 21, HASH_SEQ)])
def test_fixups_emulated(emu_ctx, k, m, kind):
    _check(emu_ctx, k, m, kind, 1500, 1, 4096)


@pytest.mark.gpu
@pytest.mark.parametrize("k,m,kind,genome,lo,hi", [(31, 15, HASH_SEQ, 1500, 1, 1000), (31, 15, HASH_SEQ, 10_000, 1000, 4096),
                                                   (45, 21, HASH_SEQ, 10_000, 500, 4096),
                                                   (63, 21, HASH_RK128, 10_000, 300, 4096),
                                                   (31, 15, HASH_SEQ, 60_000, 4097, 1 << 30),
                                                   (63, 21, HASH_RK128, 150_000, 4097, 1 << 30)])
def test_fixups(gpu_ctx, k, m, kind, genome, lo, hi):
    print(f"case fixups k={k} kind={kind} genome={genome}", flush=True)
    _check(gpu_ctx, k, m, kind, genome, lo, hi)


@pytest.mark.gpu
def test_fixups_colored(gpu_ctx):
    _check_colored(gpu_ctx, 0.002)
