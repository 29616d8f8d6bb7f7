"""Records past their unit's region: spread over the stripes of the spill list, or,
when a stripe is short, staged again into one list; records and solid table
against the oracle, with and without colors."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_SEQ, Params
from oracle import binding as O
from tests.helpers import record_tuples, solid_array

pytestmark = pytest.mark.gpu


# unit_cap 1: nearly every record spills, more than n_bytes / 64 + 65536 of them
# in the larger input; 40: some records of most units
@pytest.mark.parametrize("genome,unit_cap", [(20_000, 1), (20_000, 40), (400_000, 1), (400_000, 40)])
@pytest.mark.parametrize("colored", [False, True])
def test_spill(gpu_ctx, genome, unit_cap, colored):
    print(f"case spill genome={genome} unit_cap={unit_cap} colored={colored}", flush=True)
    k, m, b, sb = 27, 11, 4, 2
    data = synth.reads(synth.genome(141, genome), 142, genome // 12, 150, 0.005)
    gpu_ctx.set_tuning(unit_cap=unit_cap)
    try:
        if colored:
            seps = np.flatnonzero(data == 10) + 1
            starts = np.array([0, seps[seps.size // 3], seps[seps.size // 2]], np.uint64)
            colors = np.array([2, 0, 1], np.uint32)
            gpu_ctx.bucketing(data, Params(k, m, b, sb, 0, HASH_SEQ, 1), colors=(starts, colors))
            o = O.bucketing_colored(data, k, m, b, sb, starts, colors, threads=4)
        else:
            gpu_ctx.bucketing(data, Params(k, m, b, sb, 0, HASH_SEQ, 1))
            o = O.bucketing(data, k, m, b, sb, threads=4)
        assert record_tuples(gpu_ctx.records()) == record_tuples(o.records())
        gpu_ctx.kmers_merge()
        o.merge(k, b, sb, HASH_SEQ, 1, 4)
        assert np.array_equal(solid_array(gpu_ctx.solid()), solid_array(o.solid()))
    finally:
        gpu_ctx.set_tuning()
