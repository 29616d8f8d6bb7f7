"""The solid table after a merge: dense whatever the fill of the merge's output
chunks, against the oracle."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_RK128, HASH_SEQ, Params
from oracle import binding as O
from tests.helpers import bitmaps_from_sets, colored_solid_array, solid_array

pytestmark = pytest.mark.gpu


# no entry at all, less than one chunk of 4096, a few chunks, more entries than
# the wavefronts' open chunks leave free (so that entries stay and move)
@pytest.mark.parametrize("genome,k,m,kind,s", [(500, 31, 15, HASH_SEQ, 200), (900, 31, 15, HASH_SEQ, 1),
                                               (4097, 63, 21, HASH_RK128, 1), (60_000, 45, 21, HASH_SEQ, 2),
                                               (400_000, 31, 15, HASH_SEQ, 1)])
def test_dense_solid_table(gpu_ctx, genome, k, m, kind, s):
    g = synth.genome(61, genome)
    data = synth.reads(g, 62, max(8, genome // 8), 150, 0.005)
    print(f"case dense table genome={genome} k={k} kind={kind} s={s}", flush=True)
    gpu_ctx.bucketing(data, Params(k, m, 4, 2, 0, kind, s))
    gpu_ctx.kmers_merge()
    o = O.bucketing(data, k, m, 4, 2, threads=4)
    o.merge(k, 4, 2, kind, s, 4)
    got, want = solid_array(gpu_ctx.solid()), solid_array(o.solid())
    assert (want.shape[0] == 0) == (s == 200)
    assert got.shape == want.shape and np.array_equal(got, want)


def test_dense_colored_table(gpu_ctx):
    gs = synth.config3_genomes(0.01, 40)
    data, starts = synth.contigs_joined(gs, 5, 3000, 9000)
    colors = np.arange(40, dtype=np.uint32)
    gpu_ctx.bucketing(data, Params(31, 15, 4, 2, 0, HASH_SEQ, 1), colors=(starts, colors))
    gpu_ctx.kmers_merge()
    o = O.bucketing_colored(data, 31, 15, 4, 2, starts, colors, threads=4)
    o.merge(31, 4, 2, HASH_SEQ, 1, 4)
    off, cols = o.solid_colors()
    want = colored_solid_array(o.solid(), bitmaps_from_sets(off, cols, 2))
    assert np.array_equal(colored_solid_array(gpu_ctx.solid(), gpu_ctx.solid_colors()), want)
