"""Query batches cut into spans of positions, not queries: queries shorter than
k, empty ones, ones that end at or around the spans' and the 64-position steps'
edges, many in one step, long ones over several spans, N runs, unaligned
device buffers; every key kind, and color counts on both sides of the 64
lanes.  Against the oracle, emulated and on the GPU."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_RK128, HASH_SEQ, GpuContext, Params
from oracle import binding as O

KINDS = [(31, 15, HASH_SEQ, 0), (32, 12, HASH_SEQ, 0), (33, 14, HASH_SEQ, 0), (64, 21, HASH_SEQ, 0),
         (12, 6, HASH_SEQ, 0), (21, 9, HASH_RK128, 0), (63, 21, HASH_RK128, 0), (64, 21, HASH_RK128, 0),
         (31, 15, HASH_SEQ, 1), (31, 15, HASH_SEQ, 63), (45, 21, HASH_SEQ, 64), (31, 15, HASH_SEQ, 65),
         (31, 15, HASH_SEQ, 130), (45, 21, HASH_RK128, 33)]


def _queries(rng, g: np.ndarray, k: int, big: int) -> np.ndarray:
    text = g.tobytes()
    lens = [0, 1, k - 1, k, k + 1, 0, 0, 62, 63, 64, 65, 127, 128, 1023, 1024, 1025, 1024 + k, 2048 + k - 1, 3 * 1024]
    lens += list(rng.integers(0, 2 * k + 20, 60)) + list(rng.integers(0, 4, 70)) + list(rng.integers(500, 4000, big))
    out = []
    for i, n in enumerate(lens):
        a = int(rng.integers(0, max(1, len(text) - int(n))))
        q = bytearray(text[a:a + int(n)])
        if i % 4 == 1 and n > 8:
            q[int(n) // 2] = ord("N")
        if i % 5 == 2 and n > 8:
            q[3] = ord("a") if q[3] != ord("A") else ord("c")
        out.append(bytes(q) + b"\n")
    return np.frombuffer(b"".join(out), np.uint8).copy()


def _check(ctx, k, m, kind, n_colors, big, device=False):
    rng = np.random.default_rng(500 + k + n_colors)
    g = synth.genome(91, 6000)
    if n_colors:
        parts, starts = synth.contigs_joined([np.roll(g, 37 * i)[:900 + (i * 61) % 800] for i in range(n_colors)], 5,
                                             300, 900)
        colors = (starts, np.arange(n_colors, dtype=np.uint32))
        o = O.bucketing_colored(parts, k, m, 3, 2, *colors, threads=4)
    else:
        parts, colors = synth.reads(g, 92, 300, 150, 0.005), None
        o = O.bucketing(parts, k, m, 3, 2, threads=4)
    ctx.bucketing(parts, Params(k, m, 3, 2, 0, kind, 1), colors=colors)
    ctx.kmers_merge()
    ctx.index_build()
    o.merge(k, 3, 2, kind, 1, 4)
    q = _queries(rng, g, k, big)
    qk, mt, cc = o.query(q, k, kind, n_colors)
    assert int(mt.sum()) > 0
    got = [ctx.query(q)]
    if device:
        n = qk.size
        for off in (0, 1, 15):
            d_q, _ = ctx.upload(np.concatenate([np.zeros(off, np.uint8), q]))
            d_k, d_m, d_c = ctx.alloc(n * 8), ctx.alloc(n * 8), ctx.alloc(max(1, n * n_colors) * 4)
            ctx.query_device_noalloc(d_q + off, q.size, n, d_k, d_m, d_c if n_colors else None)
            got.append((ctx.download(d_k, np.zeros(n, np.uint64)), ctx.download(d_m, np.zeros(n, np.uint64)),
                        ctx.download(d_c, np.zeros((n, n_colors), np.uint32)) if n_colors else None))
            for p in (d_q, d_k, d_m, d_c):
                ctx.free(p)
    for a, b, c in got:
        assert np.array_equal(a, qk) and np.array_equal(b, mt)
        if n_colors:
            assert np.array_equal(c.astype(np.uint64), cc)


@pytest.fixture(scope="module")
def emu_ctx():
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    ctx.set_tuning(merge_wgs_per_cu=1)
    yield ctx
    ctx.close()


@pytest.mark.parametrize("k,m,kind,n_colors", KINDS)
def test_query_positions_emulated(emu_ctx, k, m, kind, n_colors):
    _check(emu_ctx, k, m, kind, n_colors, 0)


@pytest.mark.gpu
@pytest.mark.parametrize("k,m,kind,n_colors", KINDS)
def test_query_positions(gpu_ctx, k, m, kind, n_colors):
    print(f"case query positions k={k} kind={kind} colors={n_colors}", flush=True)
    _check(gpu_ctx, k, m, kind, n_colors, 20, device=True)


@pytest.mark.gpu
def test_query_positions_full_spans(gpu_ctx):
    # 9 MB of queries: spans of 1024 positions
    print("case query positions, full spans", flush=True)
    _check(gpu_ctx, 31, 15, HASH_SEQ, 0, 4000, device=True)
