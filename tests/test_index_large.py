"""Query indexes of 4 Mi entries and more of 64-bit keys, which are built by
partition: the positions they hold (a color set is read through them), on both
sides of that size, and the general build where there is no room to gather the
entries."""
import json

import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_SEQ, GpuContext, Params, colormap_write_sets

LINE = 4 << 20


@pytest.mark.gpu
@pytest.mark.parametrize("length,part", [(462_500, False), (481_250, True)])
def test_index_colors(gpu_ctx, length, part):
    print(f"case index colors length={length}", flush=True)
    n, k = 8, 31
    gs = [synth.genome(300 + i, length) for i in range(n)]
    data = np.concatenate([np.append(g, np.uint8(10)) for g in gs])
    starts = np.arange(n, dtype=np.uint64) * (length + 1)
    ids = (np.arange(n, dtype=np.uint32) * 7) % 40
    gpu_ctx.bucketing(data, Params(k, 15, 8, 4, 0, HASH_SEQ, 1), colors=(starts, ids))
    gpu_ctx.kmers_merge()
    assert (int(gpu_ctx.counters()[5]) >= LINE) == part
    gpu_ctx.index_build()
    rng = np.random.default_rng(11)
    own = rng.integers(0, n, 600)
    qs = [gs[o][a:a + int(rng.integers(k, 2500))].tobytes() + b"\n" for o, a in zip(own, rng.integers(0, length - 2500, 600))]
    kmers, matched, counts = gpu_ctx.query(np.frombuffer(b"".join(qs), np.uint8))
    assert np.array_equal(kmers, matched)
    want = np.zeros((600, int(ids.max()) + 1), np.uint64)
    want[np.arange(600), ids[own]] = kmers
    assert np.array_equal(counts.astype(np.uint64), want)


@pytest.mark.parametrize("room", [True, False])
def test_large_graph_emulated(tmp_path, monkeypatch, room):
    """A graph of two sequences, one k-mer set in color 0 and one in 0 and 2."""
    from tests.emu import build as emu_build

    k, sizes = 31, (3_000_000, 1_400_000)
    g = [synth.genome(400 + i, s) for i, s in enumerate(sizes)]
    entries = sum(s - k + 1 for s in sizes)
    assert entries >= LINE
    lib = emu_build.build()
    fa, qf = tmp_path / "graph.fa", tmp_path / "q.fa"
    fa.write_bytes(b"".join(b">%d LN:i:%d C:%x:%d\n%s\n" % (i, s, i, s - k + 1, g[i].tobytes()) for i, s in enumerate(sizes)))
    colormap_write_sets(str(tmp_path / "graph.colors.dat"), ["a", "b", "c"], [[0], [0, 2]], lib_path=lib)
    cut = [(0, 5), (1, 1_399_700), (0, 2_999_700), (1, 700_000), (0, 1_234_567)]
    qf.write_bytes(b"".join(b">q\n%s\n" % g[i][a:a + 300].tobytes() for i, a in cut))
    if not room:  # 20 bytes per entry and an eighth
        monkeypatch.setenv("GGCAT_EMU_FAIL_BYTES", f"{entries * 22}-{entries * 23}")
    ctx = GpuContext(0, lib_path=lib)
    out = ctx.query_graph(str(fa), str(qf), str(tmp_path / "out"), k, colors=True)
    ctx.close()
    got = [json.loads(line) for line in open(out)]
    assert [r["query_index"] for r in got] == list(range(len(cut)))
    assert [r["matches"] for r in got] == [{"0": 1.0} if i == 0 else {"0": 1.0, "2": 1.0} for i, _ in cut]
