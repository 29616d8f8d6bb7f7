"""Host query batches whose bytes cannot hold, or do not hold, the stated number
of records are refused before room for that many results is asked for: with 1024
colors the results of the counts below would take up to 17 TB."""
import ctypes as C

import numpy as np
import pytest

from ggcat_amd import synth
from ggcat_amd.native import EINVAL, HASH_SEQ, GpuContext, Params

LINE = 1 << 20  # bytes from which the device finds the offsets


def _check(ctx):
    g = synth.genome(51, 700)
    data = np.append(g, np.uint8(10))
    ctx.bucketing(data, Params(31, 15, 2, 1, 0, HASH_SEQ, 1),
                  colors=(np.zeros(1, np.uint64), np.array([1023], np.uint32)))
    ctx.kmers_merge()
    ctx.index_build()
    # one query of the whole genome, the rest newlines
    q = np.concatenate([data, np.full(LINE + 5 - data.size, 10, np.uint8)])
    n = q.size - 700
    out = np.full(4, 77, np.uint64)
    for count in (n - 1, n + 1, q.size, q.size + 1, 0xFFFFFFFF):
        rc = ctx.lib.ggcat_gpu_query(ctx.h, q.ctypes.data_as(C.POINTER(C.c_uint8)), q.size, count, None,
                                     out.ctypes.data_as(C.POINTER(C.c_uint64)), None)
        assert rc == EINVAL and (out == 77).all(), (count, rc)


def _check_long(ctx):
    """After _check, a batch of one query of a megabase is answered."""
    g = synth.genome(51, 700)
    q = np.concatenate([np.resize(g, LINE), np.array([10], np.uint8)])
    kmers, matched, counts = ctx.query(q)
    assert kmers.tolist() == [LINE - 30] and matched[0] >= (700 - 30) * (LINE // 700)
    assert counts[0, 1023] == matched[0] and int(counts[0, :1023].sum()) == 0


def test_query_refusals_emulated():
    from tests.emu import build as emu_build

    ctx = GpuContext(0, lib_path=emu_build.build())
    ctx.set_tuning(merge_wgs_per_cu=1)
    _check(ctx)
    ctx.close()


@pytest.mark.gpu
def test_query_refusals(gpu_ctx):
    print("case query refusals", flush=True)
    _check(gpu_ctx)
    _check_long(gpu_ctx)
