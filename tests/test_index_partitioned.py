"""The query index on both sides of the size from which entries of 64-bit keys are
gathered by partition, as large with 128-bit keys, and at a size whose partitions take
the larger bucket count: every k-mer of the graph's own sequence is found, none
of another one."""
import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import HASH_RK128, HASH_SEQ, Params

pytestmark = pytest.mark.gpu
LINE = 4 << 20  # entries from which the build is partitioned (64-bit keys)


# (a k-mer between two sub-buckets has an entry in each: about 1 + 2 / (k - m + 1) entries per base)
@pytest.mark.parametrize("k,m,kind,genome,part", [(31, 15, HASH_SEQ, 3_700_000, False), (31, 15, HASH_SEQ, 3_800_000, True),
                                                  (63, 21, HASH_RK128, 3_900_000, False),
                                                  (63, 21, HASH_RK128, 4_200_000, True),
                                                  (45, 21, HASH_SEQ, 4_300_000, True), (21, 9, HASH_SEQ, 9_000_001, True),
                                                  (31, 15, HASH_SEQ, 165_000_000, True)])
def test_index(gpu_ctx, k, m, kind, genome, part):
    print(f"case index k={k} kind={kind} genome={genome}", flush=True)
    g = synth.genome(131, genome)
    data = np.append(g, np.uint8(10))
    gpu_ctx.bucketing(data, Params(k, m, 8, 4, 0, kind, 1))
    gpu_ctx.kmers_merge()
    n = int(gpu_ctx.counters()[5])
    assert (n >= LINE) == part and (genome < 100_000_000 or n * 2 // 5 > 8192 << 13), n
    gpu_ctx.index_build()
    rng = np.random.default_rng(7)
    own = [g[a:a + int(rng.integers(k, 3000))].tobytes() + b"\n" for a in rng.integers(0, genome - 3000, 1500)]
    own += [g[:3000].tobytes() + b"\n", g[-3000:].tobytes() + b"\n"]
    qk, matched, _ = gpu_ctx.query(np.frombuffer(b"".join(own), np.uint8))
    assert np.array_equal(qk, matched) and int(qk.min()) >= 1
    if k >= 31:
        other = synth.genome(132, 2_000_000).reshape(-1, 2000)
        other = np.concatenate([other, np.full((other.shape[0], 1), 10, np.uint8)], 1).reshape(-1)
        qk, matched, _ = gpu_ctx.query(other)
        assert int(qk.min()) == 2000 - k + 1 and int(matched.sum()) == 0
