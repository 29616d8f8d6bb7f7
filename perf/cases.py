"""Workloads for timing the framework through its public entry points.

A case is a dict of plain values.  "op" says which calls one pass makes:

  table    bucketing + k-mer merge of reads in HBM; the solid table taken to
           the host and ordered by (sub-bucket, k-mer)
  screen   bucketing + merge + query index of reads in HBM, then the number of
           solid k-mers of each read of a sample of the same reads
  host     the same from reads in host memory
  files    the same from a FASTA file (build_from_files)
  colored  the same for contigs of several genomes, one color per genome, with
           the matches of each query per color
  maximal  maximal unitigs of a merged graph, taken to the host
  chains   unitigs inside each sub-bucket of a merged graph, with their flags
  query    one query batch in host memory against an indexed graph

The order of the solid table and of the unitigs is not specified, so the
passes that return them put them in a canonical order, as a program that
writes or compares them does.  Inputs are synthetic: a random genome (with
diverged repeat copies where "repeats" > 0), reads of both strands with
substitution errors, a few N bases and a share of trimmed reads.
"""
import ctypes
import os
import tempfile

import numpy as np
import torch

from ggcat_amd.native import HASH_RK128, HASH_SEQ, BuildOptions, GpuContext, plan_build

DEV = "cuda"
SAMPLE = 100_000  # reads screened per pass at most


# ---- cases -------------------------------------------------------------------

def _reads(name, op, k, m, genome, coverage, read, err, repeats=0.0, rk=False, s=2, trim=0.0, forward=False):
    return {"name": name, "op": op, "k": k, "m": m, "genome": genome, "coverage": coverage, "read": read, "err": err,
            "repeats": repeats, "rk": rk, "s": s, "trim": trim, "forward": forward}


def listed():
    return [
        # one viral genome: the smallest build, where launches and waits count
        _reads("virus-table-k31", "table", 31, 15, 30_000, 40, 150, 0.005),
        # a small genome counted with the automatic m for k = 21
        _reads("small-table-k21", "table", 21, 0, 700_000, 25, 101, 0.005, trim=0.2),
        # a bacterial isolate from its FASTA file: the reference's usual build call
        _reads("bacterium-files-k31", "files", 31, 15, 5_000_000, 30, 150, 0.005),
        # reads that arrive in host memory from a decoder
        _reads("bacterium-host-k27", "host", 27, 0, 4_000_000, 60, 150, 0.005, trim=0.2),
        # a deep eukaryotic read set resident in HBM, the benchmark's k = 31 shape
        _reads("large-screen-k31", "screen", 31, 15, 40_000_000, 40, 250, 0.01, repeats=0.2),
        # long k with rabin-karp128 keys, the benchmark's k = 63 shape
        _reads("large-screen-k63-rk", "screen", 63, 21, 30_000_000, 30, 150, 0.005, repeats=0.3, rk=True),
        # long k with 128-bit seq-hash keys (the hash unitigs need)
        _reads("medium-screen-k47", "screen", 47, 0, 8_000_000, 30, 150, 0.005, repeats=0.2),
        # a pangenome: assembled contigs, one color per genome
        {"name": "pangenome-colored-k31", "op": "colored", "k": 31, "m": 15, "genomes": 64, "genome": 700_000,
         "s": 2, "queries": 4000, "qmin": 100, "qmax": 2000},
        # the graph's maximal unitigs, what a build finally hands out
        _reads("maximal-unitigs-k31", "maximal", 31, 15, 10_000_000, 40, 250, 0.01, repeats=0.2),
        # the unitigs the merge hands to the next stage, with 128-bit keys
        _reads("bucket-unitigs-k45", "chains", 45, 21, 800_000, 30, 150, 0.005, repeats=0.2),
        # one served batch against a pangenome
        {"name": "query-colored-k31", "op": "query", "k": 31, "m": 15, "genomes": 64, "genome": 700_000, "s": 2,
         "queries": 5000, "qmin": 100, "qmax": 10_000},
        # one short request against a small uncolored graph: its latency
        {"name": "query-reads-k31", "op": "query", "k": 31, "m": 15, "genomes": 0, "genome": 1_000_000, "s": 2,
         "queries": 64, "qmin": 100, "qmax": 300},
    ]


def draw(rng):
    """One more case of the listed ones' ranges."""
    def spread(lo, hi):
        return int(round(lo * (hi / lo) ** rng.random()))

    op = rng.choice(["table", "screen", "screen", "host", "files", "colored", "maximal", "chains", "query", "query"])
    k, m, rk = rng.choice([(31, 15, False), (31, 0, False), (21, 0, False), (25, 9, False), (27, 0, False),
                           (32, 12, False), (45, 21, False), (47, 0, False), (63, 21, False), (63, 21, True),
                           (55, 0, True), (31, 15, True)])
    if op == "colored" or (op == "query" and rng.random() < 0.6):
        genomes = spread(8, 128)
        return {"op": op, "k": 31 if rng.random() < 0.7 else 27, "m": rng.choice([15, 0]), "genomes": genomes,
                "genome": spread(50_000, 700_000) * 64 // max(genomes, 64), "s": rng.choice([1, 2]),
                "queries": spread(16, 4000), "qmin": 100, "qmax": spread(300, 4000)}
    if op == "query":
        return {"op": op, "k": k, "m": m, "genomes": 0, "genome": spread(50_000, 2_000_000), "s": 1, "rk": rk,
                "queries": spread(1, 5000), "qmin": 100, "qmax": spread(150, 3000)}
    if op in ("maximal", "chains"):
        rk = False  # unitigs need seq-hash keys
    read = rng.choice([100, 101, 125, 150, 151, 250])
    if read < 1.5 * k:
        read = 150
    hi = {"table": 1_000_000, "screen": 20_000_000, "host": 4_000_000, "files": 5_000_000, "maximal": 8_000_000,
          "chains": 2_000_000}[op]
    c = _reads("", op, k, m, spread(20_000, hi), rng.randint(15, 40), read, rng.choice([0.001, 0.005, 0.01]),
               rng.choice([0.0, 0.2, 0.3]), rk, rng.choice([1, 2, 2, 3]), rng.choice([0.0, 0.2]),
               op in ("table", "screen") and rng.random() < 0.2)
    del c["name"]
    return c


# ---- inputs ------------------------------------------------------------------

_ACGTN = (65, 67, 71, 84, 78)  # codes 0..3 (complement 3 - c), 4 = N


def _letters(codes):
    return torch.tensor(_ACGTN, dtype=torch.uint8, device=DEV)[codes.to(torch.int32)]


def _substitute(codes, rate, gen):
    """Substitutions at about `rate` of the positions (in place).  A position
    drawn twice is given the same base twice."""
    n = int(codes.numel() * rate)
    if n:
        at = torch.randint(0, codes.numel(), (n,), generator=gen, device=DEV)
        by = (1 + (at * 2654435761 >> 16) % 3).to(torch.uint8)
        codes[at] = (codes[at] + by) & 3


def _genome(length, repeats, gen):
    g = torch.randint(0, 4, (length,), generator=gen, device=DEV, dtype=torch.uint8)
    unit = min(4000, max(200, length // 50))
    n = int(length * repeats) // unit
    if n and length > 2 * unit:
        # diverged copies of other stretches
        src = torch.randint(0, length - unit, (n,), generator=gen, device=DEV)
        dst = torch.randperm(length // unit, generator=gen, device=DEV)[:n] * unit
        span = torch.arange(unit, device=DEV)
        copies = g[src[:, None] + span].reshape(-1)
        _substitute(copies, 0.015, gen)
        g[(dst[:, None] + span).reshape(-1)] = copies
    return g


def _read_set(case, gen):
    """Joined reads (each followed by a newline) as a uint8 tensor in HBM, and
    the byte offset behind each of the first SAMPLE reads."""
    length, L = case["genome"], case["read"]
    g = _genome(length, case["repeats"], gen)
    n = max(1, length * case["coverage"] // L)
    span = torch.arange(L, device=DEV)
    parts = []
    step = max(1, (48 << 20) // L)
    for i in range(0, n, step):
        c = min(step, n - i)
        start = torch.randint(0, length - L + 1, (c,), generator=gen, device=DEV)
        back = torch.randint(0, 2, (c,), generator=gen, device=DEV, dtype=torch.uint8)[:, None]
        at = torch.where(back == 1, start[:, None] + (L - 1) - span, start[:, None] + span)
        r = g[at]
        r = torch.where(back == 1, 3 - r, r)
        del at
        _substitute(r.view(-1), case["err"], gen)
        flat = r.view(-1)
        flat[torch.randint(0, flat.numel(), (flat.numel() // 20_000 + 1,), generator=gen, device=DEV)] = 4
        out = torch.empty((c, L + 1), dtype=torch.uint8, device=DEV)
        out[:, :L] = _letters(r)
        out[:, L] = 10
        if case["trim"] > 0:
            # a share of the reads cut at a quality drop
            cut = torch.rand((c,), generator=gen, device=DEV) < case["trim"]
            keep = torch.where(cut, torch.randint(L // 3, L + 1, (c,), generator=gen, device=DEV), L)
            col = torch.arange(L + 1, device=DEV)
            out = out[(col < keep[:, None]) | (col == L)]
        parts.append(out.reshape(-1))
    return torch.cat(parts)


def _sample_of(joined, n):
    """(bytes, records) of the first n records of a joined tensor at most."""
    head = joined[:min(joined.numel(), n * 512)]
    ends = torch.nonzero(head == 10).flatten()[:n]
    return int(ends[-1]) + 1, int(ends.numel())


def _pangenome(case, gen, rng):
    """(joined contigs tensor, color starts, colors, genome codes)."""
    anc = _genome(case["genome"], 0.1, gen)
    parts, starts, genomes, pos = [], [], [], 0
    nl = torch.tensor([10], dtype=torch.uint8, device=DEV)
    for _ in range(case["genomes"]):
        lo = int(rng.integers(0, max(1, anc.numel() // 4)))
        own = torch.randint(0, 4, (max(1, anc.numel() // 20),), generator=gen, device=DEV, dtype=torch.uint8)
        g = torch.cat([anc[lo:].clone(), own])
        _substitute(g, 0.01, gen)
        genomes.append(g)
        starts.append(pos)
        letters, o = _letters(g), 0
        while o < letters.numel():
            e = min(letters.numel(), o + int(rng.integers(20_000, 100_001)))
            parts += [letters[o:e], nl]
            pos += e - o + 1
            o = e
    return (torch.cat(parts), np.array(starts, np.uint64), np.arange(len(starts), dtype=np.uint32), genomes)


def _queries(case, genomes, gen, rng):
    """Joined queries: lengths log-uniform in [qmin, qmax], half of them from
    the genomes with 2% substitutions, half random."""
    n, lo, hi = case["queries"], case["qmin"], case["qmax"]
    lens = np.exp(rng.uniform(np.log(lo), np.log(hi), n)).astype(np.int64)
    pool = torch.cat(genomes)
    lens = np.minimum(lens, pool.numel() - 1)
    ends = np.cumsum(lens + 1)
    total = int(ends[-1])
    own = rng.random(n) < 0.5
    first = torch.from_numpy((rng.random(n) * (pool.numel() - lens)).astype(np.int64) - (ends - lens - 1)).to(DEV)
    rec = torch.repeat_interleave(torch.arange(n, device=DEV), torch.from_numpy(lens + 1).to(DEV))
    at = (torch.arange(total, device=DEV) + first[rec]).clamp_(0, pool.numel() - 1)
    q = pool[at]
    _substitute(q, 0.02, gen)
    noise = torch.randint(0, 4, (total,), generator=gen, device=DEV, dtype=torch.uint8)
    q = _letters(torch.where(torch.from_numpy(own).to(DEV)[rec], q, noise))
    q[torch.from_numpy(ends - 1).to(DEV)] = 10
    return q


# ---- prepare -----------------------------------------------------------------

def _params(case, n_bytes):
    o = BuildOptions(case["k"], case["m"], case["s"], 0, int(case.get("forward", False)),
                     HASH_RK128 if case.get("rk") else HASH_SEQ, int(case.get("genomes", 0) > 0))
    return o, plan_build(o, n_bytes)


def prepare(case, seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    rng = np.random.default_rng(seed)
    op = case["op"]
    st = {"op": op, "case": case, "ctx": GpuContext(0)}
    if case.get("genomes", 0):
        joined, starts, colors, genomes = _pangenome(case, gen, rng)
        st["colors"] = (starts, colors)
        q = _queries(case, genomes, gen, rng)
        n_q = case["queries"]
    elif op == "query":
        g = _genome(case["genome"], 0.1, gen)
        joined = torch.cat([_letters(g), torch.tensor([10], dtype=torch.uint8, device=DEV)])
        st["s"] = 1
        q = _queries(case, [g], gen, rng)
        n_q = case["queries"]
    else:
        joined = _read_set(case, gen)
        nb, n_q = _sample_of(joined, SAMPLE)
        q = joined[:nb]
    n_bytes = int(joined.numel())
    options, params = _params(case, n_bytes)
    if op == "query" and not case.get("genomes", 0):
        params.min_multiplicity = 1  # an assembled sequence
    st.update(options=options, params=params, n_q=n_q, q_bytes=int(q.numel()))
    if op in ("table", "maximal", "chains"):
        # result buffers with room to spare
        n, k = int(3 * _solid(case)) + 4096, case["k"]
        size = {"keys": (n, 1 if k <= 32 and not case["rk"] else 2), "sub": n, "mult": n, "flags": n} \
            if op == "table" else {"seq": n * (2 + k // 8), "sub": n, "flags": n}
        of = {"keys": torch.int64, "sub": torch.int32, "mult": torch.int32, "flags": torch.uint8, "seq": torch.uint8}
        st["out"] = {name: torch.zeros(shape, dtype=of[name], device=DEV) for name, shape in size.items()}
    if op in ("table", "screen", "colored"):
        st["reads"] = joined
    if op in ("screen", "colored"):
        # device buffers of the screening results
        nc = case.get("genomes", 0)
        st["q"] = q.clone() if q.data_ptr() % 16 else q
        st["matched"] = torch.zeros(n_q, dtype=torch.int64, device=DEV)
        st["query_kmers"] = torch.zeros(n_q, dtype=torch.int64, device=DEV)
        st["color_counts"] = torch.zeros((n_q, nc), dtype=torch.int32, device=DEV) if nc else None
    if op in ("host", "files", "query"):
        st["q"] = q.cpu().numpy()
    if op == "host":
        st["reads"] = joined.cpu().numpy()
    if op == "files":
        st["dir"] = tempfile.TemporaryDirectory()
        st["path"] = os.path.join(st["dir"].name, "reads.fa")
        n_rec = int((joined == 10).sum())
        # ">\n" in front of every record
        ends = torch.nonzero(joined == 10).flatten()
        head = torch.cat([torch.zeros(1, dtype=torch.int64, device=DEV), ends[:-1] + 1]) + \
            2 * torch.arange(n_rec, device=DEV)
        fa = torch.empty(n_bytes + 2 * n_rec, dtype=torch.uint8, device=DEV)
        body = torch.ones(fa.numel(), dtype=torch.bool, device=DEV)
        body[head] = False
        body[head + 1] = False
        fa[body] = joined
        fa[head] = ord(">")
        fa[head + 1] = 10
        fa.cpu().numpy().tofile(st["path"])
    torch.cuda.synchronize()
    if op in ("maximal", "chains", "query"):
        # the graph that the program keeps
        ctx = st["ctx"]
        ctx.bucketing(None, params, colors=st.get("colors"), device_ptr=joined.data_ptr(), n_bytes=n_bytes)
        ctx.kmers_merge()
        if op == "query":
            ctx.index_build()
    return st


# ---- run ---------------------------------------------------------------------

def _counts(ctx):
    """input bytes, records, record bases, k-mer occurrences, solid entries"""
    return ctx.counters()[[0, 1, 2, 3, 5]].astype(np.int64)


def _into(out, got):
    """The results at the front of the program's buffers, zeros behind them."""
    for name, x in got.items():
        if x.shape[0] > out[name].shape[0]:
            raise RuntimeError(f"{x.shape[0]} entries of {name}: the buffer holds {out[name].shape[0]}")
        out[name][:x.shape[0]] = x
        out[name][x.shape[0]:] = 0
    return out


def _ordered_table(ctx, out):
    s = ctx.solid()
    keys = torch.from_numpy(s.keys.view(np.int64)).to(DEV)
    sub = torch.from_numpy(s.sub.view(np.int32)).to(DEV)
    order = torch.argsort(keys[:, 0], stable=True)
    order = order[torch.argsort(sub[order], stable=True)]
    return _into(out, {"keys": keys[order], "sub": sub[order],
                       "mult": torch.from_numpy(s.mult.view(np.int32)).to(DEV)[order],
                       "flags": torch.from_numpy(s.flags).to(DEV)[order]})


def _ordered_unitigs(ctx, joined, k, out):
    n, nb = ctx.unitig_counts(joined=joined)
    seq = torch.empty(nb, dtype=torch.uint8, pin_memory=True)
    sub = torch.empty(n, dtype=torch.int32, pin_memory=True)
    flags = torch.empty(n, dtype=torch.uint8, pin_memory=True)
    u8, u32 = ctypes.POINTER(ctypes.c_uint8), ctypes.POINTER(ctypes.c_uint32)
    ctx._check(ctx.lib.ggcat_gpu_unitigs_copy(ctx.h, ctypes.cast(seq.data_ptr(), u8), ctypes.cast(sub.data_ptr(), u32),
                                              ctypes.cast(flags.data_ptr(), u8)), "ggcat_gpu_unitigs_copy")
    seq, sub, flags = seq.to(DEV), sub.to(DEV), flags.to(DEV)
    ends = torch.nonzero(seq == 10).flatten()
    starts = torch.cat([ends.new_zeros(1), ends[:-1] + 1])
    order = torch.argsort(sub, stable=True)
    for lo in range(((k - 1) // 31) * 31, -1, -31):  # by the first k-mer, then the sub-bucket
        word = torch.zeros(n, dtype=torch.int64, device=DEV)
        for i in range(lo, min(k, lo + 31)):
            word = (word << 2) | ((seq[starts + i] >> 1) & 3)
        order = order[torch.argsort(word[order], stable=True)]
    size = ends - starts + 1
    size, src = size[order], starts[order]
    off = torch.cumsum(size, 0) - size
    at = torch.arange(nb, device=DEV) + torch.repeat_interleave(src - off, size, output_size=nb)
    return _into(out, {"seq": seq[at], "sub": sub[order], "flags": flags[order]})


def run(state):
    op, ctx, params = state["op"], state["ctx"], state["params"]
    if op == "query":
        qk, matched, colors = ctx.query(state["q"])
        out = {"query_kmers": qk.astype(np.int64), "matched": matched.astype(np.int64)}
        if colors is not None:
            out["color_counts"] = colors.view(np.int32)
        return out
    if op in ("maximal", "chains"):
        return _ordered_unitigs(ctx, op == "maximal", state["case"]["k"], state["out"])
    if op == "files":
        ctx.build_from_files([state["path"]], state["options"])
    else:
        reads = state["reads"]
        if op == "host":
            ctx.bucketing(reads, params)
        else:
            ctx.bucketing(None, params, colors=state.get("colors"), device_ptr=reads.data_ptr(),
                          n_bytes=reads.numel())
        ctx.kmers_merge()
    if op == "table":
        return dict(_ordered_table(ctx, state["out"]), counts=_counts(ctx))
    ctx.index_build()
    if op in ("host", "files"):
        qk, matched, _ = ctx.query(state["q"])
        return {"counts": _counts(ctx), "query_kmers": qk.astype(np.int64), "matched": matched.astype(np.int64)}
    cc = state["color_counts"]
    ctx.query_device_noalloc(state["q"].data_ptr(), state["q_bytes"], state["n_q"], state["query_kmers"].data_ptr(),
                             state["matched"].data_ptr(), cc.data_ptr() if cc is not None else None)
    out = {"counts": _counts(ctx), "query_kmers": state["query_kmers"], "matched": state["matched"]}
    if cc is not None:
        out["color_counts"] = cc
    return out


# ---- what a pass cannot do without -------------------------------------------

def _bases(case):
    if case.get("genomes", 0):
        return case["genomes"] * case["genome"]
    return case["genome"] if case["op"] == "query" else case["genome"] * case["coverage"]


def _solid(case):
    """About how many solid k-mers the graph has: the genome's, and with
    s <= 2 those with a substitution seen often enough."""
    if case["op"] == "query" or case.get("genomes", 0):
        return case["genome"]
    cov, k, e = case["coverage"], case["k"], case["err"]
    seen = {1: 1.0, 2: 0.07}.get(case["s"], 0.0)
    return case["genome"] * (1 + seen * min(1.0, k * e) * cov * (1 - k / case["read"]))


def work(case):
    """Inputs read once and outputs written once; no floating point."""
    op, key = case["op"], 8 if case["k"] <= 32 and not case.get("rk") else 16
    q_len = 0
    if "queries" in case:
        lo, hi = case["qmin"], case["qmax"]
        q_len = case["queries"] * ((hi - lo) / np.log(hi / lo) + 17 + 4 * case["genomes"])
    if op == "query":
        return {"bytes": float(q_len), "flops": 0.0}
    if op in ("maximal", "chains"):
        return {"bytes": float(_solid(case) * (key + 4 + 2)), "flops": 0.0}
    out = 0.0
    if op == "table":
        out = _solid(case) * (key + 9)
    elif op == "colored":
        out = q_len
    else:
        out = SAMPLE * (case["read"] + 17.0)
    return {"bytes": float(_bases(case) * (1 + 1 / case.get("read", 50_000)) + out), "flops": 0.0}


# ---- exact values ------------------------------------------------------------

def _kmer_codes(joined, k):
    """Canonical k-mers of a joined tensor as int64 (one exact word up to
    k = 31, else two words folded to one 64-bit fingerprint), and where a
    window holds only ACGT."""
    u = joined & 0xDF
    code = torch.full_like(joined, 4)
    for c, ch in enumerate(_ACGTN[:4]):
        code[u == ch] = c
    n = joined.numel() - k + 1
    bad = torch.zeros(joined.numel() + 1, dtype=torch.int32, device=DEV)
    torch.cumsum(code == 4, 0, dtype=torch.int32, out=bad[1:])
    ok = bad[k:] == bad[:n]
    code = (code & 3).to(torch.int64)

    def words(rc):
        got = []
        for lo in range(0, k, 31):
            w = torch.zeros(n, dtype=torch.int64, device=DEV)
            for i in range(lo, min(k, lo + 31)):
                j = k - 1 - i if rc else i
                c = code[j:j + n]
                w = (w << 2) | (3 - c if rc else c)
            got.append(w)
        return got

    fw, rc = words(False), words(True)
    less = torch.zeros(n, dtype=torch.bool, device=DEV)
    for a, b in zip(reversed(fw), reversed(rc)):
        less = (a < b) | ((a == b) & less)
    key = torch.zeros(n, dtype=torch.int64, device=DEV)
    for a, b in zip(fw, rc):
        key = key * -7046029254386353131 + torch.where(less, a, b)
    return key, ok


def exact(case, seed):
    """Per-query counts from plainly counted k-mers (seq-hash keys); None for
    the passes that return tables and unitigs, and for inputs that take long
    to sort."""
    if case["op"] in ("table", "maximal", "chains", "colored") or case.get("genomes", 0) or case.get("forward") or \
            case.get("rk") or _bases(case) > 250_000_000:
        return None
    st = prepare(dict(case, op="screen") if case["op"] != "query" else case, seed)
    k, s = case["k"], st["params"].min_multiplicity
    if case["op"] == "query":
        gen = torch.Generator(device=DEV)
        gen.manual_seed(seed)
        reads = torch.cat([_letters(_genome(case["genome"], 0.1, gen)),
                           torch.tensor([10], dtype=torch.uint8, device=DEV)])
        q = torch.from_numpy(st["q"]).to(DEV)
    else:
        reads, q = st["reads"], st["q"][:st["q_bytes"]]
    key, ok = _kmer_codes(reads, k)
    key, count = torch.unique(key[ok], return_counts=True)
    key = key[count >= s]
    qkey, qok = _kmer_codes(q, k)
    at = torch.searchsorted(key, qkey).clamp_(max=max(0, key.numel() - 1))
    hit = qok & (key[at] == qkey) if key.numel() else qok & False
    ends = torch.nonzero(q == 10).flatten()
    starts = torch.cat([ends.new_zeros(1), ends[:-1] + 1])
    sums = torch.zeros(q.numel() + 1, dtype=torch.int64, device=DEV)
    sums[1:hit.numel() + 1] = torch.cumsum(hit, 0)
    sums[hit.numel() + 1:] = sums[hit.numel()]
    out = {"query_kmers": (ends - starts - k + 1).clamp_(min=0), "matched": sums[ends] - sums[starts]}
    return out if case["op"] == "query" else dict(out, counts=None)
