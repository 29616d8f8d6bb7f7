"""Unitig paths of every length around the spacing of the splitters, long ones
(thousands of splitters), and circular ones of which the short have no splitter
on them: per sub-bucket and joined, against the oracle, emulated and on the
GPU."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_SEQ, GpuContext, Params
from oracle import binding as O
from tests.helpers import joined
from tests.test_unitigs import canon_unitigs


def _data(k: int, long: int) -> np.ndarray:
    rng = np.random.default_rng(1200 + k)
    recs = [synth.genome(int(rng.integers(1, 1 << 30)), k - 1 + n).tobytes() for n in list(range(1, 36)) + [100, 257]]
    recs.append(synth.genome(123, long).tobytes())
    for n in (40, 75, 300):  # circular sequences of n bases: cycles of n k-mers
        c = synth.genome(int(rng.integers(1, 1 << 30)), n).tobytes()
        recs.append((c * 3)[:n + k - 1])
    return joined(recs)


def _check(ctx, k, m, long):
    data = _data(k, long)
    ctx.bucketing(data, Params(k, m, 3, 1, 0, HASH_SEQ, 1))
    ctx.kmers_merge()
    o = O.bucketing(data, k, m, 3, 1, threads=4)
    o.merge(k, 3, 1, HASH_SEQ, 1, 4)
    for both in (False, True):
        want = canon_unitigs(*o.unitigs(k, joined=both))
        assert canon_unitigs(*ctx.unitigs(joined=both)) == want
        if both:
            assert max(len(s) for _, s, _ in want) >= long and sum(1 for _, _, f in want if f == 4) >= 3


@pytest.mark.parametrize("k,m", [(31, 15), (45, 21)])
def test_paths_emulated(k, m):
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    ctx.set_tuning(merge_wgs_per_cu=1)
    try:
        _check(ctx, k, m, 3000)
    finally:
        ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("k,m,long", [(31, 15, 5000), (31, 15, 400_000), (45, 21, 100_000), (32, 21, 5000)])
def test_paths(gpu_ctx, k, m, long):
    print(f"case unitig paths k={k} m={m} long={long}", flush=True)
    _check(gpu_ctx, k, m, long)
