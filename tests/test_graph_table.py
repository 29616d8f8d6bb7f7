"""A graph read from files becomes the context's table with keys (and colors)
only: what needs multiplicities, flags or sub-buckets is refused, also where the
buffers of an earlier build are large enough to be read, and the keys can be
copied."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import ESTATE, HASH_SEQ, GGCATGpuError, GpuContext, Params, _ptr, _u64p


def _check(ctx, tmp_path, built_before: bool):
    k = 31
    g = synth.genome(47, 900)
    fa, qf = tmp_path / "graph.fa", tmp_path / "query.fa"
    fa.write_bytes(b">0 LN:i:900\n" + g.tobytes() + b"\n")
    qf.write_bytes(b">q\n" + g[100:300].tobytes() + b"\n")
    if built_before:
        ctx.bucketing(synth.reads(synth.genome(48, 4000), 49, 150, 150, 0.0), Params(k, 15, 3, 1, 0, HASH_SEQ, 1))
        ctx.kmers_merge()
        assert ctx.solid().mult.size > 900
    ctx.query_graph(str(fa), str(qf), str(tmp_path / "out"), k)
    keys = np.zeros((900 - k + 1, 1), np.uint64)
    null = [None] * 3
    assert ctx.lib.ggcat_gpu_solid_copy(ctx.h, _ptr(keys, _u64p), *null) == 0
    code = ((np.frombuffer(g.tobytes(), np.uint8) >> 1) & 3).astype(object)
    want = []
    for i in range(900 - k + 1):
        fw = sum(int(code[i + j]) << (2 * j) for j in range(k))
        rc = sum((int(code[i + j]) ^ 2) << (2 * (k - 1 - j)) for j in range(k))
        want.append(min(fw, rc))
    assert sorted(int(x) for x in keys[:, 0]) == sorted(want)
    for call in (ctx.solid, ctx.unitig_counts, lambda: ctx.unitig_counts(joined=True)):
        with pytest.raises(GGCATGpuError, match=rf"status {ESTATE}\b"):
            call()
    # the next build's table is whole again
    ctx.bucketing(np.append(g, np.uint8(10)), Params(k, 15, 3, 1, 0, HASH_SEQ, 1))
    ctx.kmers_merge()
    assert np.unique(ctx.solid().keys).size == len(set(want))
    assert ctx.unitig_counts(joined=True)[0] == 1


@pytest.mark.parametrize("built_before", [False, True])
def test_graph_table_emulated(tmp_path, built_before):
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    ctx.set_tuning(merge_wgs_per_cu=1)
    _check(ctx, tmp_path, built_before)
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("built_before", [False, True])
def test_graph_table(tmp_path, built_before):
    print(f"case graph table built_before={built_before}", flush=True)
    ctx = GpuContext(0)
    _check(ctx, tmp_path, built_before)
    ctx.close()
