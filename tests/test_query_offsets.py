"""Host query batches around the size from which their offsets are found on the
device: the same counts as the oracle's on both sides, empty queries and a
block of newlines among them, and batches whose bytes are not the stated number
of records refused as before."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_SEQ, GGCATGpuError, Params
from oracle import binding as O

pytestmark = pytest.mark.gpu
K, M = 31, 15
LINE = 1 << 20  # bytes from which the device finds the offsets


@pytest.fixture(scope="module")
def graph(gpu_ctx):
    g = synth.genome(95, 20_000)
    data = synth.reads(g, 96, 2000, 150, 0.005)
    o = O.bucketing(data, K, M, 3, 2, threads=4)
    o.merge(K, 3, 2, HASH_SEQ, 1, 4)
    return g, data, o


def _batch(g, n_bytes):
    """n_bytes of queries, a run of empty ones across a counting block's end."""
    rng = np.random.default_rng(n_bytes)
    text = g.tobytes()
    out, size = [], 0
    while size < n_bytes:
        n = int(rng.integers(0, 400))
        if 16_000 < size < 16_500:
            out.append(b"\n" * 700)
        else:
            a = int(rng.integers(0, len(text) - n))
            out.append(text[a:a + n] + b"\n")
        size += len(out[-1])
    q = np.frombuffer(b"".join(out), np.uint8)[:n_bytes].copy()
    q[-1] = 10
    return q


@pytest.mark.parametrize("n_bytes", [LINE - 1, LINE, LINE + 1, LINE + 16_383, 2 * LINE + 7])
def test_query_offsets(gpu_ctx, graph, n_bytes):
    g, data, o = graph
    print(f"case query offsets n_bytes={n_bytes}", flush=True)
    gpu_ctx.bucketing(data, Params(K, M, 3, 2, 0, HASH_SEQ, 1))
    gpu_ctx.kmers_merge()
    gpu_ctx.index_build()
    q = _batch(g, n_bytes)
    qk, mt, _ = o.query(q, K, HASH_SEQ, 0)
    a, b, _ = gpu_ctx.query(q)
    assert int(mt.sum()) > 0 and np.array_equal(a, qk) and np.array_equal(b, mt)
    lib, n = gpu_ctx.lib, int((q == 10).sum())
    import ctypes

    u8, u64 = ctypes.POINTER(ctypes.c_uint8), ctypes.POINTER(ctypes.c_uint64)
    got = np.full(n + 1, 77, np.uint64)
    for count, cut in ((n - 1, 0), (n + 1, 0), (n, 1)):
        bad = np.ascontiguousarray(q[:q.size - cut] if not cut else np.append(q[:-1], np.uint8(65)))
        rc = lib.ggcat_gpu_query(gpu_ctx.h, bad.ctypes.data_as(u8), bad.size, count, got.ctypes.data_as(u64),
                                 got.ctypes.data_as(u64), None)
        assert rc == 1 and (got == 77).all()
    with pytest.raises(GGCATGpuError):
        gpu_ctx.query(np.append(q[:-1], np.uint8(65)))
    assert np.array_equal(gpu_ctx.query(q)[1], mt)
