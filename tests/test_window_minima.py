"""Window minima of the staging pass for every kind of window width w = k - m:
the block sizes 2, 4, 8 and 16 at the ends of their ranges, windows over one to
three whole blocks, and w == 16 with windows too long for the 64-bit slice of
its own variant.  Records against the oracle, emulated and on the GPU."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_SEQ, GpuContext, Params
from oracle import binding as O
from tests.helpers import edge_records_inline, inline_capacity, joined, record_tuples

# w:     2        3       4         5        7        8        9         11        15        16
CASES = [(5, 3), (9, 6), (13, 9), (64, 59), (15, 8), (20, 12), (31, 22), (21, 10), (47, 32), (63, 47),
         # 17     31        32        33        42        47        48        49        62       63
         (32, 15), (45, 14), (48, 16), (47, 14), (63, 21), (60, 13), (64, 16), (63, 14), (64, 2), (64, 1)]


def _inputs(k: int, m: int) -> np.ndarray:
    rng = np.random.default_rng(9000 + 67 * k + m)
    cap = inline_capacity(k, m)
    recs = []
    g = synth.genome(71, 6000)
    reads = synth.reads(g, 72, 60, 150, 0.01).tobytes().split(b"\n")[:-1]
    for r in edge_records_inline(rng, k)[:30] + reads + [g[:3100].tobytes()]:
        # records longer than a slot (the long-record pool) stay off the GPU
        o = O.bucketing(joined([r]), k, m, 4, 2, threads=1).records()["length"]
        if o.size == 0 or int(o.max()) <= cap:
            recs.append(r)
    return joined(recs)


def _check(ctx, k, m):
    data = _inputs(k, m)
    want = O.bucketing(data, k, m, 4, 2, threads=2).records()
    assert want["sub"].size > 100
    ctx.bucketing(data, Params(k, m, 4, 2, 0, HASH_SEQ, 1))
    assert record_tuples(ctx.records()) == record_tuples(want)


@pytest.fixture(scope="module")
def emu_ctx():
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    yield ctx
    ctx.close()


@pytest.mark.parametrize("k,m", CASES)
def test_window_widths_emulated(emu_ctx, k, m):
    _check(emu_ctx, k, m)


@pytest.mark.gpu
@pytest.mark.parametrize("k,m", CASES)
def test_window_widths(gpu_ctx, k, m):
    print(f"case window width k={k} m={m} w={k - m}", flush=True)
    _check(gpu_ctx, k, m)
