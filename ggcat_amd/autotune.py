"""Schedule autotuner for the build: times bucketing + merge of a sample
under candidate schedules (ggcat_gpu_set_tuning knobs) and keeps the
fastest.  The knobs change which kernel path and table size handle a work
item, never the result; every candidate's solid table is checked against the
first one's digest.  Choices are cached per (k, m, hash, colored).

The bucket count (-b) changes the result (MapEntries are per sub-bucket), so
it is only searched when the caller allows it, and then returned as a
recommendation alongside the schedule.
"""
from __future__ import annotations

import itertools
import json
import os
from dataclasses import asdict, dataclass, replace

import numpy as np

from .native import Params

KNOBS = ("item_occ", "lds_max_occ", "merge_wgs_per_cu", "part_occ", "lds_table_log", "table_pct", "no_dedup",
         "unit_bytes", "use_graphs", "unit_cap", "rec_cap",
         "merge_threads")


@dataclass
class Schedule:
    item_occ: int = 0
    unit_bytes: int = 0
    table_pct: int = 0
    lds_table_log: int = 0
    no_dedup: int = 0
    merge_wgs_per_cu: int = 0
    use_graphs: int = 0
    rec_cap: int = 0
    unit_cap: int = 0
    merge_threads: int = 0

    def apply(self, ctx) -> None:
        ctx.set_tuning(item_occ=self.item_occ, unit_bytes=self.unit_bytes, table_pct=self.table_pct, lds_table_log=self.lds_table_log,
                       no_dedup=self.no_dedup, merge_wgs_per_cu=self.merge_wgs_per_cu, use_graphs=self.use_graphs,
                       rec_cap=self.rec_cap, unit_cap=self.unit_cap, merge_threads=self.merge_threads)


def unit_log(n_bytes: int, n_sub: int, unit_bytes: int) -> int:
    """log2 of the physical units per sub-bucket: the sub-bucket's share of the
    input is halved until it is at most unit_bytes (ggcat_gpu_bucketing's rule)."""
    xb = 0
    while xb < 10 and (n_bytes >> xb) // n_sub > unit_bytes and n_sub << (xb + 1) <= 1 << 25:
        xb += 1
    return xb


def unit_size(n_bytes: int, n_sub: int, unit_bytes: int) -> int:
    """Bytes of a physical unit of an input; many values of unit_bytes come to
    the same units."""
    return (n_bytes >> unit_log(n_bytes, n_sub, unit_bytes)) // n_sub


def n_sub(params: Params) -> int:
    return ((1 << params.buckets_log) + 1) << params.second_buckets_log


def sample_params(params: Params, full_bytes: int, sample_bytes: int) -> Params:
    """The parameters with fewer sub-buckets, as the sample is smaller, so that
    its sub-buckets have as many units of the same size as the full input's: a
    work item is a run of units of one sub-bucket, and with too few of them
    large items would not fill up on the sample as they do on the full input."""
    less = max(0, round(np.log2(full_bytes / max(sample_bytes, 1))))
    s = min(less, params.second_buckets_log)
    b = min(less - s, params.buckets_log - 1)
    return Params(params.k, params.m, params.buckets_log - b, params.second_buckets_log - s, params.forward_only,
                  params.hash_kind, params.min_multiplicity)


def sample_fraction(full_bytes: int, cap: int) -> float:
    """The share of an input of full_bytes that a sample of at most cap bytes
    should hold: a power of two, which gives the same unit sizes."""
    j = 0
    while full_bytes / 2**j > cap:
        j += 1
    return 1 / 2**j


def default_item_occ(k: int, lds: int) -> int:
    """Occurrences per work item that the merge takes by default with a table of
    lds entries: half of it, three quarters with two-word keys."""
    return lds // 4 * 3 if 32 < k < 64 else lds // 2


def default_grid(k: int) -> list[Schedule]:
    """Unit size x record-table size x LDS table size: the knobs whose best
    value depends on the input (coverage, error rate, k); the others are
    fixed at values that measured best on every configuration tried.  Units
    below 2000 bytes are tried for k > 32 only: their counters and open lines
    stay in cache on a sample and do not on a large input (4 Gbases, k = 31:
    staging 33.1 ms with units of 956 bytes, 22.7 with 1913), and it is k <= 32
    whose records are many."""
    logs = (11,) if k <= 32 else (10,)
    sizes = (2000, 3000) if k <= 32 else (1400, 2000, 3000)
    out = []
    for ub, rc, lg in itertools.product(sizes, (256, 512), logs):
        out.append(Schedule(unit_bytes=ub, table_pct=200, lds_table_log=lg, rec_cap=rc, use_graphs=1))
    # smaller tables over small units, in workgroups of 128 and 256 threads
    # (more resident workgroups per CU)
    small = sizes[0]
    out.append(Schedule(unit_bytes=small, table_pct=200, lds_table_log=lg - 1, rec_cap=128, use_graphs=1,
                        merge_threads=128))
    for rc in (128, 256):
        out.append(Schedule(unit_bytes=small, table_pct=200, lds_table_log=lg - 1, rec_cap=rc, use_graphs=1,
                            merge_threads=256))
    return out


def load_grid(best: Schedule, k: int) -> list[Schedule]:
    """Second stage around the best first-stage schedule: the hash table's
    load factor (table slots per 100 k-mer occurrences of a work item) and
    the work-item size, which together set how full the LDS tables run."""
    lds = 1 << (best.lds_table_log or (11 if k <= 32 else 10))
    out = []
    if k <= 32:  # identical records counted once, each distinct record rolled by one thread
        s = Schedule(**asdict(best))
        s.no_dedup = 2
        out.append(s)
    for pct, occ in itertools.product((100, 200, 400), (lds // 2, lds, 2 * lds)):
        if (pct, occ) == (best.table_pct or 200, best.item_occ or default_item_occ(k, lds)):
            continue
        s = Schedule(**asdict(best))
        s.table_pct, s.item_occ = pct, occ
        out.append(s)
    return out


def _digest(ctx) -> tuple:
    s = ctx.solid()
    keys = s.keys.astype(np.uint64)
    with np.errstate(over="ignore"):
        # every key word is mixed in (2-word keys for k > 32 and rabin-karp128)
        kh = np.zeros(keys.shape[0], np.uint64)
        for j in range(keys.shape[1]):
            kh = (kh ^ keys[:, j]) * np.uint64(0x9E3779B97F4A7C15)
            kh ^= kh >> np.uint64(29)
        h = kh ^ (s.sub.astype(np.uint64) << np.uint64(32)) \
            ^ (s.mult.astype(np.uint64) << np.uint64(8)) ^ s.flags.astype(np.uint64)
        return int(s.mult.size), int(np.bitwise_xor.reduce(h)) if h.size else 0, int(h.sum(dtype=np.uint64))


def autotune(ctx, sample: np.ndarray, params: Params, grid: list[Schedule] | None = None, repeats: int = 3,
             cache_path: str | None = None, colored: bool = False, bucket_logs: tuple[int, ...] = (),
             min_gain: float = 0.02, full_bytes: int | None = None) -> dict:
    """Times schedules on `sample`, for inputs of full_bytes (the sample's own
    size when not given): each runs with the units and sub-buckets that it
    comes to on the full input (sample_params, and the nearest unit size), since
    a table that suits units of 1000 bytes may split most items of units of
    2000; schedules that come to the same units there are tried once.  Returns
    {"schedule": Schedule fields, "ms": best bucketing+merge ms on the sample,
    "tried": n, "buckets_log": recommended b}; applies the best schedule to
    ctx.  A schedule is timed by the device (the bucketing's
    kernels and the merge call between its stream events, the lowest of
    `repeats` runs), so host-side call overheads, which do not grow with the
    input, do not decide between schedules on a small sample; a schedule
    must be at least `min_gain` faster than the best so far to replace it (a
    schedule's time on a 250 MB sample differs by 2 % between runs)."""
    key = f"k{params.k}-m{params.m}-h{params.hash_kind}-c{int(colored)}"
    if cache_path and os.path.exists(cache_path):
        cached = json.load(open(cache_path)).get(key)
        if cached:
            Schedule(**cached["schedule"]).apply(ctx)
            return cached
    two_stage = grid is None
    grid = grid or default_grid(params.k)
    sample = np.ascontiguousarray(sample, np.uint8)
    full = full_bytes or sample.size

    def distinct(schedules):
        """The first of the schedules that differ in unit_bytes only and come to
        the same units on the full input."""
        out = {}
        for s in schedules:
            unit = unit_size(full, n_sub(params), s.unit_bytes) if s.unit_bytes else 0
            out.setdefault((unit, *(v for f, v in asdict(s).items() if f != "unit_bytes")), s)
        return list(out.values())

    def time_on_sample(sch, p):
        """Device milliseconds of bucketing and merge with the schedule for p,
        with the sample's unit size nearest to the full input's."""
        q = sample_params(p, full, sample.size)
        sizes = {(sample.size >> x) // n_sub(q) for x in range(11)} - {0}
        if sch.unit_bytes and sizes:
            want = max(unit_size(full, n_sub(p), sch.unit_bytes), 1)
            sch = replace(sch, unit_bytes=min(sizes, key=lambda u: abs(np.log(u / want))))
        sch.apply(ctx)
        ctx.bucketing(None, q, device_ptr=ptr, n_bytes=n)
        ctx.kmers_merge()
        tm = ctx.timings()
        return float(tm[5] + tm[6])

    ptr, n = ctx.upload(sample)
    ref = None
    best = None
    tried = 0

    def run(sch):
        nonlocal ref, best, tried
        ts = [time_on_sample(sch, params) for _ in range(repeats)]
        d = _digest(ctx)
        if ref is None:
            ref = d
        elif d != ref:
            raise RuntimeError(f"schedule {sch} changed the solid table")
        tried += 1
        ms = min(ts)
        # a later schedule replaces the best only when it is at least
        # min_gain faster: of schedules within the sample's timing noise of
        # each other the one timed first is kept (the second stage times the
        # first stage's best before its variations)
        if best is None or ms < best[0] * (1.0 - min_gain):
            best = (ms, sch)

    try:
        for sch in distinct(grid):
            run(sch)
        if two_stage:
            for sch in load_grid(best[1], params.k):
                run(sch)
        rec_b = params.buckets_log
        for b in bucket_logs:
            p2 = Params(params.k, params.m, b, params.second_buckets_log, params.forward_only, params.hash_kind,
                        params.min_multiplicity)
            ms = time_on_sample(best[1], p2)
            if ms < best[0]:
                rec_b = b
    finally:
        ctx.free(ptr)
    best[1].apply(ctx)
    out = {"schedule": asdict(best[1]), "ms": round(best[0], 3), "tried": tried, "buckets_log": rec_b,
           "sample_bytes": int(sample.size)}
    if cache_path:
        allc = json.load(open(cache_path)) if os.path.exists(cache_path) else {}
        allc[key] = out
        json.dump(allc, open(cache_path, "w"), indent=1)
    return out
