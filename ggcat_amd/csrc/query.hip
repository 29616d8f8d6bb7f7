// query.hip -- colored / uncolored k-mer queries against the solid k-mer
// table of the last merge, kept resident in HBM.
//
// Semantics (crates/querier/src/pipeline/parallel_kmers_query.rs:372-471,
// counters_sorting.rs:106-273, colored_query_output.rs:200-320,
// crates/querier/src/lib.rs:138-150): every k-mer occurrence of an ACGT run
// of a query whose canonical hash is a graph k-mer counts once for the query
// and once for each color of that k-mer's color set.  The graph k-mer set is
// the solid table of the build (the k-mers of its unitigs).
//
// Index: a hash table of 4-entry buckets (KmerTable) over the solid entries;
// an entry holds its key words and its position in the solid arrays, so a
// lookup reads one line in most cases.
#include "common.h"

namespace gg {

GG_DEV uint64_t mix64(uint64_t x) {
    x ^= x >> 30;
    x *= 0xbf58476d1ce4e5b9ULL;
    x ^= x >> 27;
    x *= 0x94d049bb133111ebULL;
    x ^= x >> 31;
    return x;
}

GG_DEV uint64_t index_hash(uint64_t lo, uint64_t hi) { return mix64(lo ^ mix64(hi + 0x9E3779B97F4A7C15ULL)); }

constexpr uint32_t NO_POS = 0xFFFFFFFFu;

// Hash table of solid entries: nb buckets of 4 entries, a bucket's entries in
// arrival order, the first free one empty (position NO_POS); an entry whose
// bucket is full goes to the next bucket with room.  Entry words: 64-bit keys
// {key, position}, 128-bit keys {low, high, position, 0}, so a bucket is 64 or
// 128 bytes.  1.6 slots per entry: few buckets overflow (mean fill 2.5).
// Bound by one random counter update and one random 16-byte store per entry
// (the counters of 100 M entries fit the 256 MiB cache); building it takes one
// pass over the keys where offsets of exactly sized buckets took a counting
// pass, a scan and a placing pass with its own atomics, and a lookup reads the
// bucket alone instead of offsets, keys and positions.  Index of 57.7 M
// entries 8.3 -> 5.9 ms (0.4 of it clearing).
struct KmerTable {
    ulonglong2* slots;  // [nb * 4 * key_words]
    uint32_t* count;  // [nb] entries that arrived (more than 4: the bucket overflowed); not used by the partitioned build
    uint32_t nb;
    uint32_t key_words;
};

constexpr uint32_t TAB_BUCKET = 4;
__host__ __device__ inline uint32_t table_buckets(uint64_t n) { return (uint32_t)(n * 2 / 5 + 1); }

GG_DEV uint32_t table_bucket(const KmerTable& T, uint64_t lo, uint64_t hi) {
    return (uint32_t)(((index_hash(lo, hi) >> 32) * T.nb) >> 32);
}

// Entries [0, n) of the solid keys into the table (cleared: counts 0, slots ~0).
__global__ void table_insert_kernel(KmerTable T, const uint64_t* key, uint64_t n) {
    for (uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; p < n; p += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t lo = key[p * T.key_words], hi = T.key_words == 2 ? key[p * 2 + 1] : 0;
        uint32_t b = table_bucket(T, lo, hi), r;
        // 4 nb > n: some bucket has room
        while ((r = atomicAdd(&T.count[b], 1u)) >= TAB_BUCKET) b = b + 1 == T.nb ? 0 : b + 1;
        ulonglong2* e = T.slots + ((uint64_t)b * TAB_BUCKET + r) * T.key_words;
        ulonglong2 v;
        v.x = lo;
        v.y = T.key_words == 1 ? p : hi;
        e[0] = v;
        if (T.key_words == 2) {
            v.x = p;
            v.y = 0;
            e[1] = v;
        }
    }
}

// ---- large tables of 64-bit keys ------------------------------------------------
// Random counter updates and random 16-byte stores reach 27 and 22 G/s on this
// memory, and 10 to 16 G/s each when mixed.  From PART_MIN entries on they are
// kept apart and local: entries are first gathered by partition (2^shift
// neighbouring buckets), where a workgroup reserves room for its share of a
// partition with one update, then a workgroup per partition counts its buckets'
// entries in LDS and stores into a span of 0.5 MB (1 MB), all spans in flight
// fitting the 256 MiB cache.  It also writes the free slots, so the table is
// not cleared first.  Index of 57.7 M entries 5.95 -> 2.9 ms, of 4.9 M 0.34 ->
// 0.25 ms.  128-bit keys stay with the general build, whose entries are one
// 32-byte store there: 28.9 M entries 2.0 ms against 2.35 gathered, 7 M 0.5
// against 0.6.
constexpr uint64_t PART_MIN = 4u << 20;
constexpr uint32_t PART_MAX = 8192;  // partitions (LDS counters of the gathering kernels)
constexpr uint32_t PART_EACH = 16;  // entries per thread and step of the gathering kernel, 1024 threads
constexpr uint32_t PART_SHIFT_MAX = 14;  // 16384 bucket counters are 64 KB of LDS

// Shift of the partitioned build for a table of nb buckets, 0: the general one.
__host__ __device__ inline uint32_t part_shift(uint64_t n, uint32_t nb, uint32_t key_words) {
    if (n < PART_MIN || key_words != 1) return 0;
    for (uint32_t s = 13; s <= PART_SHIFT_MAX; s++)
        if (((nb - 1) >> s) < PART_MAX) return s;
    return 0;
}

// Entries per partition (cleared before).
__global__ __launch_bounds__(1024) void part_count_kernel(KmerTable T, const uint64_t* key, uint64_t n, uint32_t shift,
                                                          uint32_t n_part, uint32_t* counts) {
    __shared__ uint32_t c[PART_MAX];
    for (uint32_t i = threadIdx.x; i < n_part; i += blockDim.x) c[i] = 0;
    __syncthreads();
    for (uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; p < n; p += (uint64_t)gridDim.x * blockDim.x)
        atomicAdd(&c[table_bucket(T, key[p], 0) >> shift], 1u);
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n_part; i += blockDim.x)
        if (c[i]) atomicAdd(&counts[i], c[i]);
}

// Entries {key, position} gathered by partition: partition q's at
// off[q] ... in any order; cursor (cleared) counts what is reserved.
__global__ __launch_bounds__(1024) void part_gather_kernel(KmerTable T, const uint64_t* key, uint64_t n, uint32_t shift,
                                                           uint32_t n_part, const uint64_t* off, uint32_t* cursor,
                                                           ulonglong2* out) {
    __shared__ uint32_t c[PART_MAX];  // entries of this step, then their start behind off
    constexpr uint64_t STEP = 1024 * PART_EACH;
    for (uint64_t p0 = blockIdx.x * STEP; p0 < n; p0 += gridDim.x * STEP) {
        for (uint32_t i = threadIdx.x; i < n_part; i += blockDim.x) c[i] = 0;
        __syncthreads();
        // partition (13 bits) << 16 | rank in the step (at most 2^14)
        uint32_t at[PART_EACH];
#pragma unroll
        for (uint32_t j = 0; j < PART_EACH; j++) {
            const uint64_t p = p0 + j * 1024 + threadIdx.x;
            at[j] = 0;
            if (p < n) {
                const uint32_t q = table_bucket(T, key[p], 0) >> shift;
                at[j] = q << 16 | atomicAdd(&c[q], 1u);
            }
        }
        __syncthreads();
        for (uint32_t i = threadIdx.x; i < n_part; i += blockDim.x)
            if (c[i]) c[i] = atomicAdd(&cursor[i], c[i]);
        __syncthreads();
#pragma unroll
        for (uint32_t j = 0; j < PART_EACH; j++) {
            const uint64_t p = p0 + j * 1024 + threadIdx.x;
            if (p < n) {
                const uint32_t q = at[j] >> 16;
                ulonglong2 v;
                v.x = key[p];
                v.y = p;
                out[off[q] + c[q] + (at[j] & 0xFFFFu)] = v;
            }
        }
        __syncthreads();  // c is cleared for the next step
    }
}

// One workgroup per partition: its entries to their buckets, the free slots
// after them; entries that overflow past the partition's last bucket go to
// `rest` (their index in `in`).
__global__ __launch_bounds__(1024) void part_insert_kernel(KmerTable T, uint32_t shift, const uint64_t* off,
                                                           const ulonglong2* in, uint32_t* rest, unsigned int* n_rest) {
    extern __shared__ __align__(16) uint8_t lds[];
    uint32_t* cnt = reinterpret_cast<uint32_t*>(lds);
    const uint32_t b0 = blockIdx.x << shift, left = T.nb - b0, nb = left < (1u << shift) ? left : 1u << shift;
    for (uint32_t i = threadIdx.x; i < nb; i += blockDim.x) cnt[i] = 0;
    __syncthreads();
    const uint64_t end = off[blockIdx.x + 1];
    for (uint64_t i = off[blockIdx.x] + threadIdx.x; i < end; i += blockDim.x) {
        const ulonglong2 v = in[i];
        uint32_t b = table_bucket(T, v.x, 0) - b0, r = TAB_BUCKET;
        while (b < nb && (r = atomicAdd(&cnt[b], 1u)) >= TAB_BUCKET) b++;
        if (b >= nb) {
            rest[atomicAdd(n_rest, 1u)] = (uint32_t)i;
            continue;
        }
        T.slots[(uint64_t)(b0 + b) * TAB_BUCKET + r] = v;
    }
    __syncthreads();
    ulonglong2 free_slot;
    free_slot.x = free_slot.y = ~0ULL;
    for (uint32_t i = threadIdx.x; i < nb * TAB_BUCKET; i += blockDim.x) {
        if (i % TAB_BUCKET >= cnt[i / TAB_BUCKET]) T.slots[(uint64_t)b0 * TAB_BUCKET + i] = free_slot;
    }
}

// The entries left over (about one per partition) from the first bucket behind
// their partition on; a slot belongs to who claims its position word.
__global__ void part_rest_kernel(KmerTable T, uint32_t shift, const ulonglong2* in, const uint32_t* rest,
                                 const unsigned int* n_rest) {
    const uint32_t n = *n_rest;
    for (uint32_t j = blockIdx.x * blockDim.x + threadIdx.x; j < n; j += gridDim.x * blockDim.x) {
        const ulonglong2 v = in[rest[j]];
        uint32_t b = table_bucket(T, v.x, 0);
        b = ((b >> shift) + 1) << shift;
        if (b >= T.nb) b = 0;
        // 4 nb > n: some bucket has room
        for (bool placed = false; !placed; b = b + 1 == T.nb ? 0 : b + 1) {
            for (uint32_t s = 0; s < TAB_BUCKET && !placed; s++) {
                ulonglong2* e = T.slots + (uint64_t)b * TAB_BUCKET + s;
                if (atomicCAS(reinterpret_cast<unsigned long long*>(&e->y), ~0ULL, (unsigned long long)v.y) != ~0ULL)
                    continue;
                e->x = v.x;
                placed = true;
            }
        }
    }
}

// Calls found(position) for the entries of a key until it returns true.
template <class F>
GG_DEV void table_find(const KmerTable& T, uint64_t lo, uint64_t hi, F&& found) {
    uint32_t b = table_bucket(T, lo, hi);
    // at most nb buckets, of which at least one is not full
    while (true) {
        const ulonglong2* e = T.slots + (uint64_t)b * TAB_BUCKET * T.key_words;
        if (T.key_words == 1) {
            ulonglong2 v[TAB_BUCKET];
#pragma unroll
            for (uint32_t i = 0; i < TAB_BUCKET; i++) v[i] = e[i];
#pragma unroll
            for (uint32_t i = 0; i < TAB_BUCKET; i++) {
                if ((uint32_t)v[i].y == NO_POS) return;
                if (v[i].x == lo && found((uint32_t)v[i].y)) return;
            }
        } else {
            for (uint32_t i = 0; i < TAB_BUCKET; i++) {
                const ulonglong2 v = e[2 * i];
                const uint32_t pos = (uint32_t)e[2 * i + 1].x;
                if (pos == NO_POS) return;
                if (v.x == lo && v.y == hi && found(pos)) return;
            }
        }
        b = b + 1 == T.nb ? 0 : b + 1;
    }
}

struct QueryArgs {
    const uint8_t* seq;  // joined queries
    uint64_t n;  // bytes in seq
    const uint64_t* qoff;  // [n_queries + 1] start of each query (query q ends at qoff[q+1] - 1, its '\n')
    uint32_t n_queries;
    uint32_t k;
    uint32_t span;  // k-mer start positions per wavefront (a multiple of 64, at most QUERY_SPAN)
    KmerTable index;
    const uint32_t* out_colors;  // color_words per solid position (colored)
    uint32_t color_words;  // 0: uncolored
    uint32_t n_colors;  // per-query color counters written (<= 32 * color_words)
    uint64_t* matched;  // [n_queries], cleared
    uint32_t* color_counts;  // [n_queries * n_colors], cleared
    const u128_t* rk_tri;  // rabin-karp128: terms of three bases per entry (see MergeArgs)
};
constexpr uint32_t QUERY_SPAN = 1024;

GG_DEV uint32_t index_lookup(const QueryArgs& A, uint64_t lo, uint64_t hi) {
    uint32_t pos = NO_POS;
    table_find(A.index, lo, hi, [&](uint32_t p) {
        pos = p;
        return true;
    });
    return pos;
}

GG_DEV uint32_t ascii_code(uint8_t c) { return (c >> 1) & 3u; }
GG_DEV bool ascii_acgt(uint8_t c) {
    const uint8_t u = c & 0xDF;
    return u == 'A' || u == 'C' || u == 'G' || u == 'T';
}

// One wavefront per `span` consecutive byte positions of the batch, whatever
// the queries' lengths: every position is the start of a k-mer, 64 at a time,
// one per lane.  The bytes become 2-bit codes and invalid / newline bits in
// LDS once; a k-mer is cut out of them (a newline is an invalid base, so none
// crosses queries), its key looked up, and the hits of the 64 positions are
// counted per query by ballots, one global atomic per query and wavefront.
// Colors: a run of neighbouring hits with the same color set (its head found by
// comparing with the lane before) is added to the wavefront's counters by all
// lanes at once, lane c taking colors c, c + 64, ...
// One workgroup per query gave a 150 bp read 120 of 256 lanes, each of which
// loaded k bytes one by one, and rabin-karp128 2 k dependent 128-bit multiplies
// per lane.  Bound by the lookups (one random line of the table each).
// 100 K reads: of 250 bp, k = 31, 2.25 -> 0.81 ms; of 150 bp, k = 63
// rabin-karp128, 3.99 -> 1.01 ms; 5000 colored queries of 100 - 10000 bp 0.64
// -> 0.44 ms.
// KIND 0: seq-hash k <= 32, 1: seq-hash k > 32, 2: rabin-karp128.
template <int KIND>
__global__ __launch_bounds__(64) void query_kernel(QueryArgs A) {
    extern __shared__ __align__(16) uint8_t lds[];
    uint32_t* counts = reinterpret_cast<uint32_t*>(lds);  // [n_colors] of the current query
    // 16 positions per chunk: the span, up to 15 bytes before it, k - 1 behind
    // it, and chunks that the reads of whole words run into
    constexpr uint32_t CHUNKS = (15 + QUERY_SPAN + 63 + 15) / 16 + 6;
    __shared__ uint32_t pk[CHUNKS];
    __shared__ uint32_t inv[CHUNKS / 2 + 1], nl[CHUNKS / 2 + 1];
    const uint32_t k = A.k, lane = threadIdx.x;
    const uint64_t p0 = (uint64_t)blockIdx.x * A.span;
    const uint32_t n_pos = A.n - p0 < A.span ? (uint32_t)(A.n - p0) : A.span;
    const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(A.seq + p0) & 15);  // chunks are 16-byte aligned
    const uint32_t n_chunks = (mis + n_pos + k - 1 + 15) / 16;
    for (uint32_t c = lane; c < n_chunks + 6; c += 64) {
        const int64_t a = (int64_t)p0 - mis + 16 * (int64_t)c;
        uint32_t packed = 0, bad = 0, ends = 0;
        if (c < n_chunks && a >= 0 && a + 16 <= (int64_t)A.n) {
            const uint4 v = *reinterpret_cast<const uint4*>(A.seq + a);
            const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
            for (uint32_t i = 0; i < 16; i++) {
                const uint8_t ch = (uint8_t)(w[i >> 2] >> (8 * (i & 3)));
                packed |= ascii_code(ch) << (2 * i);
                bad |= (ascii_acgt(ch) ? 0u : 1u) << i;
                ends |= (ch == '\n' ? 1u : 0u) << i;
            }
        } else {
            for (uint32_t i = 0; i < 16; i++) {
                const uint8_t ch =
                    c < n_chunks && a + i >= 0 && a + i < (int64_t)A.n ? A.seq[a + i] : (uint8_t)0;
                packed |= ascii_code(ch) << (2 * i);
                bad |= (ascii_acgt(ch) ? 0u : 1u) << i;
                ends |= (ch == '\n' ? 1u : 0u) << i;
            }
        }
        pk[c] = packed;
        reinterpret_cast<uint16_t*>(inv)[c] = (uint16_t)bad;
        reinterpret_cast<uint16_t*>(nl)[c] = (uint16_t)ends;
    }
    for (uint32_t c = lane; c < A.n_colors; c += 64) counts[c] = 0;
    // the query holding the first position: the last one starting at or before
    // it, 64 candidates per step
    uint32_t q = 0;
    for (uint32_t hi = A.n_queries; hi - q > 1;) {
        const uint32_t step = (hi - q + 63) / 64;
        const uint64_t at = q + (uint64_t)(lane + 1) * step;
        const uint32_t m = (uint32_t)__popcll(__ballot(at < hi && A.qoff[at] <= p0));
        q += m * step;
        hi = hi - q < step ? hi : q + step;
    }
    __syncthreads();
    uint32_t cnt = 0;  // hits of query q so far
    auto flush = [&]() {
        if (!cnt) return;
        if (lane == 0) atomicAdd(reinterpret_cast<unsigned long long*>(&A.matched[q]), (unsigned long long)cnt);
        for (uint32_t c = lane; c < A.n_colors; c += 64) {
            if (counts[c]) atomicAdd(&A.color_counts[(uint64_t)q * A.n_colors + c], counts[c]);
            counts[c] = 0;
        }
        cnt = 0;
    };
    for (uint32_t i0 = 0; i0 < n_pos; i0 += 64) {
        const uint32_t i = i0 + lane, r = mis + i;
        uint32_t pos = NO_POS;
        bool end = false;
        if (i < n_pos) {
            end = (nl[r >> 5] >> (r & 31)) & 1;
            if ((bits64(inv, r) & (~0ULL >> (64 - k))) == 0) {
                uint64_t lo, hi = 0;
                bool fwd;
                if (KIND == 0) {
                    lo = kmer_at(pk, r, k, &fwd);
                } else {
                    u128_t fw, rc;
                    kmer_pair_at(pk, r, k, &fw, &rc);
                    const u128_t key = KIND == 2 ? rk_of_kmer(A.rk_tri, k, fw, &fwd) : fw < rc ? fw : rc;
                    lo = (uint64_t)key;
                    hi = (uint64_t)(key >> 64);
                }
                pos = index_lookup(A, lo, hi);
            }
        }
        const uint64_t hits = __ballot(pos != NO_POS), ends = __ballot(end);
        uint64_t heads = 0;
        if (A.color_words) {
            // a hit whose color set is that of the hit one position before
            // continues its run
            bool same = lane && pos != NO_POS && ((hits >> (lane - 1)) & 1);
            for (uint32_t w = 0; w < A.color_words; w++) {
                const uint32_t x = pos != NO_POS ? A.out_colors[(uint64_t)pos * A.color_words + w] : 0u;
                if (lane_prev32(x) != x) same = false;
            }
            heads = __ballot(pos != NO_POS && !same);
        }
        // the 64 positions' queries in turn
        uint64_t left = ~0ULL, e = ends;
        while (true) {
            const uint64_t upto = e ? e ^ (e - 1) : ~0ULL;  // positions up to the next newline
            const uint64_t part = left & upto;
            cnt += (uint32_t)__popcll(hits & part);
            for (uint64_t h = heads & part; h; h &= h - 1) {
                const uint32_t b = (uint32_t)__builtin_ctzll(h);
                const uint64_t more = b == 63 ? 0 : (hits & ~heads) >> (b + 1);  // hits that continue the run
                const uint32_t len = 1 + (uint32_t)__builtin_ctzll(~more);
                const uint32_t hp = (uint32_t)__shfl((int)pos, (int)b);
                for (uint32_t c = lane; c < A.n_colors; c += 64)
                    counts[c] += ((A.out_colors[(uint64_t)hp * A.color_words + (c >> 5)] >> (c & 31)) & 1u) * len;
            }
            if (!e) break;
            flush();
            q++;
            left = ~upto;
            e &= e - 1;
        }
    }
    flush();
}

}  // namespace gg
