// merge.hip -- per-sub-bucket canonical k-mer counting on gfx950.
//
// Restates, per sub-bucket (bucket x second bucket, the unit of one
// kmers_transform job, crates/kmers_transform/src/lib.rs:277-386):
//   crates/assembler_kmers_merge/src/unitigs_extender/hashmap.rs:361-431
//     add_sequence: per k-mer occurrence, count += multiplicity and
//     flags |= (begin_ignored << !fw) | (end_ignored << fw)
//   crates/structs/src/map_entry.rs:79-83
//     multiplicity = count >> (flags == INCL_BEGIN|INCL_END)
//   hashmap.rs:134-137 solid filter: multiplicity >= min_multiplicity
// k-mer keys: crates/hashes/src/base/cn_seqhash_base.rs:22-72 (canonical
// 2-bit seq-hash, u64 for k <= 32, u128 for k <= 64) or
// crates/hashes/src/base/cn_rkhash_base.rs:65-110 (rabin-karp128).
//
// Work items are runs of physical units of one sub-bucket.  A k-mer shared by
// two groups of the same sub-bucket stored in different work items is seen
// half in each: both halves carry the same counter (every occurrence of such
// a k-mer is a group boundary, so it appears once on each side) and one flag
// bit each.  Those entries carry a cross mark and are combined afterwards
// (flags ORed), which yields exactly the sub-bucket's MapEntry.
//
// Table entry value: bits 0..28 counter, bit 29 cross mark, bits 30..31 the
// two MapEntry flags; one u32 atomicAdd + atomicOr update an entry.
#include "common.h"

namespace gg {

constexpr uint64_t EMPTY64 = ~0ULL;
constexpr uint32_t CNT_MASK = 0x1FFFFFFFu;
constexpr uint32_t VAL_CROSS = 1u << 29;

struct WorkItem {
    uint32_t u0;  // first physical unit
    uint32_t dup;  // 1: a unit of the item may still hold identical records (not deduplicated by the compaction)
    uint32_t occ;  // k-mer occurrences
    uint32_t sub;  // sub-bucket
    uint64_t r0, r1;  // its slots [r0, r1)
};

// One pass over a work item restricted to the k-mers whose partition hash
// falls in `part` of 2^log_parts.  Items whose distinct k-mers do not fit one
// LDS table are processed as several such passes.
struct PartWork {
    uint32_t item;
    uint32_t part;
    uint32_t log_parts;
    uint32_t occ;  // the item's k-mer occurrences (set on redo entries)
};
constexpr uint32_t MAX_LOG_PARTS = 16;

struct MergeArgs {
    const uint32_t* slots;
    uint32_t slot_words;
    const uint32_t* pool;
    uint32_t k;
    uint32_t min_mult;
    uint32_t kind;  // 0 = canonical seq-hash, 1 = canonical rabin-karp128
    uint32_t key_words;  // 1 (u64 keys) or 2 (u128 keys)
    uint32_t lds_cap;  // table entries in LDS (power of two)
    uint32_t lds_try;  // first pass: items with more occurrences go straight to partitioned passes
    uint32_t table_pct;  // table slots per 100 occurrences of a whole-item pass (power-of-two rounded)
    uint32_t dedup;  // identical records of an entry are inserted once with their count
    uint32_t rec_lds_off;  // byte offset of the record table in dynamic LDS
    uint32_t rec_cap;  // record table slots
    uint32_t rec_direct;  // items without dup: records placed in the record table by position, not hashed
    uint32_t claim;  // work entries claimed per atomic on the work cursor
    const WorkItem* items;
    const PartWork* parts;  // null: first pass, one work entry per item
    uint32_t n_work;  // entries of this pass
    unsigned int* work;  // work-stealing cursor
    PartWork* redo;  // work entries whose table overflowed (at most n_work)
    unsigned int* redo_count;
    uint64_t* out_key;  // key_words per entry, chunked (see OUT_CHUNK)
    uint32_t* out_val;  // multiplicity | flags << 30
    uint32_t* out_sub;
    unsigned int* chunk_cursor;
    uint32_t* chunk_fill;
    uint32_t n_chunks;
    uint64_t* fix_key;  // cross-marked entries awaiting their other half
    uint32_t* fix_val;
    uint32_t* fix_sub;
    unsigned long long* fix_cursor;
    uint64_t fix_cap;
    uint64_t pool_words;  // valid words in the long-record pool
    uint32_t* error_flag;  // bit 1: malformed slot
    // colored builds: per-slot color, color bitmap words per entry (0 when
    // uncolored), and the bitmaps of the output and fixup entries
    const uint32_t* slot_color;
    uint32_t color_words;
    uint32_t* out_colors;
    uint32_t* fix_colors;
    // rabin-karp128 constants (crates/hashes/src/cn_rkhash.rs:65-78)
    u128_t rk_mult, rk_mult_inv, rk_rmmult;
    u128_t rk_fwd[4], rk_bkw[4];
    u128_t rk_fwd_rm[4], rk_bkw_rm[4];  // rk_fwd[c] * rk_rmmult, rk_bkw[c] * rk_rmmult
    // per base position i < k - 1 of a k-mer and base c: entry 2(4i + c) is
    // rk_fwd[c] * rk_mult^(k-2-i), entry 2(4i + c) + 1 is rk_bkw[c] * rk_mult^(i+1)
    const u128_t* rk_pos;
    // sums of three bases' terms of a whole k-mer's two hashes: entry
    // 2(64g + c) is sum of rk_fwd[c_j] * rk_mult^(k-1-i) over the bases i =
    // 3g + j (j < 3, i < k, c_j the j-th 2-bit code of c), entry
    // 2(64g + c) + 1 the sum of rk_bkw[c_j] * rk_mult^i
    const u128_t* rk_tri;
};

GG_DEV uint32_t hash128(uint64_t lo, uint64_t hi) { return tab_hash64(lo ^ (hi * 0x9E3779B97F4A7C15ULL)); }

// Kernel variants.  MODE 0 reads every switch from the arguments: the paths
// without spread k-mers (no_dedup), k = 64, slots of 16 words and colored
// rabin-karp128.  The others have their key width, hash and colors compiled
// in, which keeps the other paths' code out of their register allocation:
//   1 seq-hash k <= 32, 4-word slots      2 seq-hash k <= 32
//   3 rabin-karp128 k <= 32               4 seq-hash 32 < k < 64
//   5 rabin-karp128 32 < k < 64           6, 7 as 2 and 4 with colors
// All of them count the canonical 2-bit k-mers, which name the same entries as
// their rabin-karp128 hashes (up to hash collisions, 2^-128 per pair of
// k-mers); an entry's hash is formed when it is emitted (rk_of_kmer), so that
// the 128-bit multiplies of the rolling hash are not paid per occurrence.
template <int MODE>
struct Mode {
    static constexpr bool FAST = MODE != 0;
    static constexpr uint32_t TKW = (MODE == 4 || MODE == 5 || MODE == 7) ? 2u : 1u;  // table key words (MODE != 0)
    static constexpr bool RK = MODE == 3 || MODE == 5;
    static constexpr bool COL = MODE == 6 || MODE == 7;
    // k-mers of a distinct record that one thread takes: one where the tags of
    // every k-mer position fit beside the other LDS tables (4-word slots: 18
    // per record at most), else runs of four, rolled
    static constexpr uint32_t SEG = MODE == 1 ? 1u : 4u;
    static GG_DEV uint32_t key_words(const MergeArgs& A) { return RK || TKW == 2 ? 2u : FAST ? 1u : A.key_words; }
    static GG_DEV uint32_t color_words(const MergeArgs& A) { return FAST && !COL ? 0u : A.color_words; }
    static GG_DEV bool dedup(const MergeArgs& A) { return FAST || A.dedup; }
    static GG_DEV uint32_t slot_words(const MergeArgs& A) { return MODE == 1 ? 4u : A.slot_words; }
    static constexpr uint32_t MAX_SW = MODE == 1 ? 4u : 8u;  // register copies of a slot
};

// Table keys of 32 < k < 64: the low 63 bits of the 2-bit k-mer and the rest,
// so that neither word is EMPTY64.
GG_DEV void pair_of(uint64_t lo, uint64_t hi, uint64_t& a, uint64_t& b) {
    a = lo & ~(1ULL << 63);
    b = (lo >> 63) | (hi << 1);
}
GG_DEV uint32_t pair_hash(uint64_t a, uint64_t b) { return tab_hash64(a ^ (b * 0x9E3779B97F4A7C15ULL)); }

// Insert one occurrence.  Returns 1 when this call claimed a new slot, 0 when
// the key was present, 2 when no slot was found within min(mask+1,
// probe_limit) probes.
template <class KP, class VP>
GG_DEV uint32_t tab_insert64(KP keys, VP vals, uint32_t mask, uint64_t key, uint32_t bits, uint32_t probe_limit,
                             uint32_t& slot) {
    uint32_t i = tab_hash64(key) & mask;
    uint32_t claimed = 0;
    for (uint32_t probes = 0;; probes++) {
        if (probes > mask || probes >= probe_limit) return 2;
        uint64_t cur = keys[i];
        if (cur == key) break;
        if (cur == EMPTY64) {
            uint64_t old = atomicCAS((unsigned long long*)&keys[i], (unsigned long long)EMPTY64,
                                     (unsigned long long)key);
            if (old == EMPTY64) {
                claimed = 1;
                break;
            }
            if (old == key) break;
        }
        i = (i + 1) & mask;
    }
    atomicAdd((uint32_t*)&vals[i], bits & CNT_MASK);
    if (bits & ~CNT_MASK) atomicOr((uint32_t*)&vals[i], bits & ~CNT_MASK);
    slot = i;
    return claimed;
}

// Two-word keys, interleaved: a slot belongs to the first key whose first word
// claims word 0 and whose second word then claims word 1.  Words only ever
// change from EMPTY64 to their value, so a key that loses either claim moves
// on and no lane waits for another; a slot costs one 16-byte read and, when
// free, two compare-and-swaps.
GG_DEV uint32_t tab_insert_pair(uint64_t* keys, uint32_t* vals, uint32_t mask, uint32_t h, uint64_t a, uint64_t b,
                                uint32_t bits, uint32_t probe_limit, uint32_t& slot) {
    uint32_t i = h & mask;
    uint32_t claimed = 0;
    for (uint32_t probes = 0;; probes++) {
        if (probes > mask || probes >= probe_limit) return 2;
        ulonglong2 cur = *reinterpret_cast<const ulonglong2*>(keys + 2 * i);
        if (cur.x == EMPTY64) {
            cur.x = atomicCAS((unsigned long long*)&keys[2 * i], (unsigned long long)EMPTY64, (unsigned long long)a);
            if (cur.x == EMPTY64) cur.x = a;
        }
        if (cur.x == a) {
            if (cur.y == EMPTY64) {
                cur.y = atomicCAS((unsigned long long*)&keys[2 * i + 1], (unsigned long long)EMPTY64,
                                  (unsigned long long)b);
                if (cur.y == EMPTY64) {
                    claimed = 1;
                    break;
                }
            }
            if (cur.y == b) break;
        }
        i = (i + 1) & mask;
    }
    atomicAdd(&vals[i], bits & CNT_MASK);
    if (bits & ~CNT_MASK) atomicOr(&vals[i], bits & ~CNT_MASK);
    slot = i;
    return claimed;
}

// 128-bit keys: a slot is claimed through its state word (0 free, 1 being
// written, 2 ready).  The loop body runs the writer and the waiters in the
// same iteration, so lanes of one wavefront cannot wait on each other; the
// wait on a slot in state 1 is bounded.
template <class KP, class SP, class VP>
GG_DEV uint32_t tab_insert128(KP klo, KP khi, SP st, VP vals, uint32_t mask, uint64_t lo, uint64_t hi,
                              uint32_t bits, uint32_t probe_limit, uint32_t& slot) {
    uint32_t i = hash128(lo, hi) & mask;
    uint32_t claimed = 0, probes = 0, spins = 0;
    bool done = false;
    while (!done) {
        uint32_t s = __hip_atomic_load((uint32_t*)&st[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        if (s == 0) {
            if (atomicCAS((uint32_t*)&st[i], 0u, 1u) == 0u) {
                klo[i] = lo;
                khi[i] = hi;
                __threadfence_block();  // the table is in LDS: workgroup scope
                atomicExch((uint32_t*)&st[i], 2u);
                claimed = 1;
                done = true;
            }
        } else if (s == 2) {
            uint64_t a = __hip_atomic_load((uint64_t*)&klo[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            uint64_t b = __hip_atomic_load((uint64_t*)&khi[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            if (a == lo && b == hi) {
                done = true;
            } else {
                i = (i + 1) & mask;
                if (++probes > mask || probes >= probe_limit) return 2;
            }
        } else if (++spins > (1u << 20)) {
            return 2;
        }
    }
    atomicAdd((uint32_t*)&vals[i], bits & CNT_MASK);
    if (bits & ~CNT_MASK) atomicOr((uint32_t*)&vals[i], bits & ~CNT_MASK);
    slot = i;
    return claimed;
}

// Rabin-karp128 hashes (cn_rkhash_base.rs:65-110) of the k-mers with index
// [i0, i1) of packed bases bw; cb(lo, hi, is_forward, idx).  The state over
// the first k - 1 bases of k-mer i0, fh = sum fwd[c] M^(k-2-i) and
// bk = sum bkw[c] M^(i+1) over its base offsets i (what the Horner loops of
// the reference's init compute), is summed from the per-position table:
// independent loads and 128-bit adds instead of two chains of k - 1
// dependent 128-bit multiplies; then each k-mer is one rolling step.
template <class CB>
GG_DEV void rk_segment(const MergeArgs& A, const uint32_t* bw, uint32_t i0, uint32_t i1, CB&& cb) {
    const uint32_t k = A.k;
    auto code = [&](uint32_t i) -> uint32_t { return (bw[i >> 4] >> (2 * (i & 15))) & 3; };
    u128_t fh = 0, bk = 0;
    for (uint32_t i = 0; i + 1 < k; i++) {
        const u128_t* e = A.rk_pos + 2 * (4 * i + code(i0 + i));
        fh += e[0];
        bk += e[1];
    }
    for (uint32_t x = i0; x < i1; x++) {
        const uint32_t in = code(x + k - 1), out = code(x);
        const u128_t cur_f = fh * A.rk_mult + A.rk_fwd[in];
        fh = cur_f - A.rk_fwd_rm[out];
        const u128_t cur_b = bk * A.rk_mult_inv + A.rk_bkw_rm[in];
        bk = cur_b - A.rk_bkw[out];
        const u128_t key = cur_f < cur_b ? cur_f : cur_b;
        cb((uint64_t)key, (uint64_t)(key >> 64), cur_f < cur_b, x);
    }
}

// Rabin-karp128 key of a k-mer from its 2-bit form x: the sums of its bases'
// terms, three bases per table entry (43 KB at k = 63: lines of one
// group are shared by the lanes), and the smaller of the two; *swap when that
// is the hash of the reverse complement.
GG_DEV u128_t rk_of_kmer(const u128_t* tri, uint32_t k, u128_t x, bool* swap) {
    u128_t f = 0, b = 0;
    for (uint32_t g = 0; 3 * g < k; g++) {
        const u128_t* e = tri + 2 * (64 * g + ((uint32_t)x & 63u));
        f += e[0];
        b += e[1];
        x >>= 6;
    }
    *swap = f > b;
    return f < b ? f : b;
}

// Iterate the k-mers of one slot; cb(lo, hi, is_forward, idx, last_idx).
template <int MODE, class CB>
GG_DEV void for_each_kmer(const MergeArgs& A, const uint32_t* slot, CB&& cb) {
    const uint32_t meta = slot[0];
    const uint32_t* bw;
    uint32_t len;
    if (meta & META_LONG) {
        len = slot[1];
        uint64_t off = (uint64_t)slot[2] | ((uint64_t)slot[3] << 32);
        if (off + ((uint64_t)len + 15) / 16 > A.pool_words) {
            atomicOr(A.error_flag, 2u);
            return;
        }
        bw = A.pool + off;
    } else {
        len = meta_len(meta);
        if (len > (Mode<MODE>::slot_words(A) - 1) * 16) {
            atomicOr(A.error_flag, 2u);
            return;
        }
        bw = slot + 1;
    }
    const uint32_t k = A.k;
    if (len < k) return;
    const uint32_t last = len - k;
    if (Mode<MODE>::FAST ? Mode<MODE>::TKW == 1 : A.kind == 0 && k <= 32) {
        const uint64_t mask = (k == 32) ? ~0ULL : ((1ULL << (2 * k)) - 1);
        uint64_t fw = 0, rc = 0;
        uint32_t word = 0;
        for (uint32_t i = 0; i < len; i++) {
            if ((i & 15) == 0) word = bw[i >> 4];
            uint64_t c = (word >> (2 * (i & 15))) & 3;
            fw = (fw >> 2) | (c << (2 * (k - 1)));
            rc = ((rc << 2) | (c ^ 2)) & mask;
            if (i + 1 >= k) cb(fw < rc ? fw : rc, 0ULL, fw < rc, i + 1 - k, last);
        }
    } else if (Mode<MODE>::FAST || A.kind == 0) {
        const u128_t mask = (k == 64) ? ~(u128_t)0 : (((u128_t)1 << (2 * k)) - 1);
        u128_t fw = 0, rc = 0;
        uint32_t word = 0;
        for (uint32_t i = 0; i < len; i++) {
            if ((i & 15) == 0) word = bw[i >> 4];
            u128_t c = (word >> (2 * (i & 15))) & 3;
            fw = (fw >> 2) | (c << (2 * (k - 1)));
            rc = ((rc << 2) | (c ^ 2)) & mask;
            if (i + 1 >= k) {
                u128_t key = fw < rc ? fw : rc;
                cb((uint64_t)key, (uint64_t)(key >> 64), fw < rc, i + 1 - k, last);
            }
        }
    } else {
        rk_segment(A, bw, 0, last + 1,
                   [&](uint64_t lo, uint64_t hi, bool fwd, uint32_t x) { cb(lo, hi, fwd, x, last); });
    }
}

// Value bits contributed by one occurrence (count 1, flags, cross mark).
GG_DEV uint32_t occurrence_bits(uint32_t meta, bool is_fwd, uint32_t idx, uint32_t last) {
    const uint32_t rflags = meta_flags(meta);
    bool begin_ignored = (rflags & 1) == 0 && idx == 0;
    bool end_ignored = (rflags & 2) == 0 && idx == last;
    uint32_t fl = ((begin_ignored ? 1u : 0u) << (is_fwd ? 0 : 1)) | ((end_ignored ? 1u : 0u) << (is_fwd ? 1 : 0));
    bool cross = (idx == 0 && (meta & META_XBEGIN)) || (idx == last && (meta & META_XEND));
    return 1u | (cross ? VAL_CROSS : 0u) | (fl << 30);
}

// Output is written in chunks of OUT_CHUNK entries.  Each wavefront owns one
// open chunk at a time (reserved with one atomic), fills it without any
// workgroup barrier and records its fill count when it moves on, so solid
// entries cost no global atomics.  Entries of chunk c live at
// [c * OUT_CHUNK, c * OUT_CHUNK + fill[c]) until out_close_holes_kernel makes
// the table dense.
constexpr uint32_t OUT_CHUNK = 4096;

// A wavefront's open chunk; every lane holds the same values.
struct EmitState {
    uint32_t chunk;  // open chunk, ~0u when none
    uint32_t fill;
};

GG_DEV void close_chunk(const MergeArgs& A, EmitState& es) {
    if ((threadIdx.x & 63) == 0 && es.chunk != ~0u && es.chunk < A.n_chunks) A.chunk_fill[es.chunk] = es.fill;
    es.chunk = ~0u;
    es.fill = 0;
}

// Emit solid entries among the table slots listed in `claimed` (n of them);
// cross-marked entries holding only one flag bit go to the fixup list.
// Wavefronts take 64 listed slots at a time.
template <int MODE>
GG_DEV void emit_solid(const MergeArgs& A, uint32_t sub, const uint64_t* klo, const uint64_t* khi, const uint32_t* st,
                       const uint32_t* vals, const uint32_t* cbits, const uint16_t* claimed, uint32_t n, EmitState& es) {
    const uint32_t W = Mode<MODE>::color_words(A), KW = Mode<MODE>::key_words(A);
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint64_t below = (1ULL << lane) - 1;
    for (uint32_t i0 = wave * 64; i0 < n; i0 += blockDim.x) {
        const uint32_t j = i0 + lane;
        const uint32_t i = j < n ? claimed[j] : 0u;
        bool solid = false, fix = false;
        uint32_t outv = 0;
        if (j < n) {
            bool occupied = Mode<MODE>::FAST || ((KW == 1) ? (klo[i] != EMPTY64) : (st[i] == 2));
            if (occupied) {
                uint32_t v = vals[i];
                uint32_t cnt = v & CNT_MASK, fl = v >> 30;
                uint32_t mult = cnt >> (fl == 3 ? 1 : 0);
                solid = mult >= A.min_mult;
                fix = solid && (v & VAL_CROSS) && (fl == 1 || fl == 2);
                outv = mult | (fl << 30);
            }
        }
        uint64_t lo = 0, hi = 0;
        if (solid) {
            if (Mode<MODE>::FAST && Mode<MODE>::TKW == 2) {
                const uint64_t a = klo[2 * i], b = klo[2 * i + 1];
                lo = a | (b << 63);
                hi = b >> 1;
            } else {
                lo = klo[i];
                if (!Mode<MODE>::FAST && KW == 2) hi = khi[i];
            }
            if (Mode<MODE>::RK) {
                bool swap;
                const u128_t key = rk_of_kmer(A.rk_tri, A.k, ((u128_t)hi << 64) | lo, &swap);
                lo = (uint64_t)key;
                hi = (uint64_t)(key >> 64);
                // the flags face the hash's strand
                if (swap) outv = (outv & 0x3FFFFFFFu) | ((outv >> 31) << 30) | ((outv & (1u << 30)) << 1);
            }
        }
        const bool main = solid && !fix;
        const uint64_t bal = __ballot(main), balf = __ballot(fix);
        const uint32_t cnt = (uint32_t)__popcll(bal);
        if (cnt) {
            if (es.chunk == ~0u || es.fill + cnt > OUT_CHUNK) {
                close_chunk(A, es);
                uint32_t c = 0;
                if (lane == 0) c = atomicAdd(A.chunk_cursor, 1u);
                es.chunk = __shfl(c, 0);
            }
            if (main && es.chunk < A.n_chunks) {
                const uint64_t pos = (uint64_t)es.chunk * OUT_CHUNK + es.fill + __popcll(bal & below);
                if (KW == 1) {
                    A.out_key[pos] = lo;
                } else {
                    A.out_key[2 * pos] = lo;
                    A.out_key[2 * pos + 1] = hi;
                }
                A.out_val[pos] = outv;
                A.out_sub[pos] = sub;
                for (uint32_t q = 0; q < W; q++) A.out_colors[pos * W + q] = cbits[i * W + q];
            }
            es.fill += cnt;
        }
        if (balf) {
            unsigned long long basef = 0;
            if (lane == 0) basef = atomicAdd(A.fix_cursor, (unsigned long long)__popcll(balf));
            basef = __shfl(basef, 0);
            if (fix) {
                uint64_t pos = basef + __popcll(balf & below);
                if (pos < A.fix_cap) {
                    if (KW == 1) {
                        A.fix_key[pos] = lo;
                    } else {
                        A.fix_key[2 * pos] = lo;
                        A.fix_key[2 * pos + 1] = hi;
                    }
                    A.fix_val[pos] = outv;
                    A.fix_sub[pos] = sub;
                    for (uint32_t q = 0; q < W; q++) A.fix_colors[pos * W + q] = cbits[i * W + q];
                }
            }
        }
    }
}

// rabin-karp128 variants: the slots of `claimed` holding solid entries, listed
// in `solid` (at most n), so that the hashes are formed by full wavefronts.
// Returns how many.
GG_DEV uint32_t list_solid(const MergeArgs& A, const uint32_t* vals, const uint16_t* claimed, uint32_t n,
                           uint16_t* solid, uint32_t* n_solid) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (uint32_t i0 = wave * 64; i0 < n; i0 += blockDim.x) {
        const uint32_t j = i0 + lane;
        const uint32_t i = j < n ? claimed[j] : 0u;
        bool is = false;
        if (j < n) {
            const uint32_t v = vals[i];
            is = ((v & CNT_MASK) >> ((v >> 30) == 3 ? 1 : 0)) >= A.min_mult;
        }
        const uint64_t bal = __ballot(is);
        if (!bal) continue;
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(n_solid, (uint32_t)__popcll(bal));
        base = __shfl(base, 0);
        if (is) solid[base + (uint32_t)__popcll(bal & ((1ULL << lane) - 1))] = (uint16_t)i;
    }
    __syncthreads();
    return *n_solid;
}

// Inserts every occurrence of the item's records whose k-mer lies in the
// work entry's partition (bits 16.. of the table hash; the slot index uses
// the low bits).  An insert that needs more than `probe_limit` probes sets
// *overflow and insertion stops (the entry is then redone as finer parts).
GG_DEV void insert_item(const MergeArgs& A, uint64_t r0, uint64_t r1, const PartWork& w, uint64_t* klo, uint64_t* khi,
                        uint32_t* st, uint32_t* vals, uint32_t* cbits, uint32_t mask, uint32_t probe_limit, uint32_t* overflow,
                        uint16_t* claimed, uint32_t* n_claimed) {
    const uint32_t W = A.color_words, KW = A.key_words;
    const uint32_t SW = A.slot_words;
    const uint32_t part_mask = (1u << w.log_parts) - 1;
    for (uint64_t r = r0 + threadIdx.x; r < r1; r += blockDim.x) {
        const uint32_t* slot = A.slots + r * SW;
        const uint32_t meta = slot[0];
        const uint32_t color = W ? A.slot_color[r] : 0u;
        const uint32_t extra = meta_mult(meta) - 1;  // identical copies stored once
        for_each_kmer<0>(A, slot, [&](uint64_t lo, uint64_t hi, bool is_fwd, uint32_t idx, uint32_t last) {
            if (*(volatile uint32_t*)overflow) return;
            if (part_mask) {
                const uint32_t h = (KW == 1) ? tab_hash64(lo) : hash128(lo, hi);
                if (((h >> 16) & part_mask) != w.part) return;
            }
            uint32_t bits = occurrence_bits(meta, is_fwd, idx, last) + extra, at = 0;
            uint32_t res = (KW == 1)
                               ? tab_insert64(klo, vals, mask, lo, bits, probe_limit, at)
                               : tab_insert128(klo, khi, st, vals, mask, lo, hi, bits, probe_limit, at);
            if (res == 2) {
                atomicOr(overflow, 1u);
                return;
            }
            if (res == 1) claimed[atomicAdd(n_claimed, 1u)] = (uint16_t)at;
            if (W) atomicOr(&cbits[at * W + (color >> 5)], 1u << (color & 31));
        });
    }
}

// ---- identical-record path -------------------------------------------------
// The reference merges identical super-k-mers of a bucket before counting
// (crates/minimizer_bucketing/src/compactor.rs:128-196, multiplicities
// summed, :159-163); counting each distinct record once with its multiplicity
// gives the same MapEntries.  Records are keyed by their whole slot (meta
// word with length, flags, minimizer position and cross marks, then the
// packed bases) plus their color; a record the table cannot take is counted
// on its own.  After deduplication every thread takes k-mers of the distinct
// records (MODE != 0), so the k-mer work is spread evenly over the workgroup.
// Record table slots (a power of two, 16..512); chunks of rec_cap / 2
// records are deduplicated at a time.  512 would cost one of the four
// workgroups that a CU's LDS holds: merge of 1.57 G occurrences (k = 31)
// 11.0 ms against 8.6 ms with 256, of 551 M (k = 63) 14.3 against 11.4 ms.
constexpr uint32_t REC_CAP_DEFAULT = 256;

struct RecTable {
    uint32_t* key;  // rec_cap * SW
    uint32_t* cnt;
    uint32_t* state;  // 0 free, 1 being written, 2 ready
    uint32_t* col;
    uint32_t* n;  // [1]: k-mers of the chunk, [2..5]: wave totals of the scan
    uint16_t* rec_of;  // each segment of SEG k-mers of the chunk: record slot << 7 | index of the segment in the record
};

// k-mers of one inline record at most.
__host__ __device__ inline uint32_t rec_max_kmers(uint32_t slot_words, uint32_t k) {
    return (slot_words - 1) * 16 >= k ? (slot_words - 1) * 16 - k + 1 : 0;
}

GG_DEV RecTable rec_table(const MergeArgs& A, uint8_t* lds) {
    RecTable R;
    uint32_t* b = reinterpret_cast<uint32_t*>(lds + A.rec_lds_off);
    R.key = b;
    b += A.rec_cap * A.slot_words;
    R.cnt = b;
    b += A.rec_cap;
    R.state = b;
    b += A.rec_cap;
    R.col = b;  // colored builds only
    if (A.color_words) b += A.rec_cap;
    R.n = b;
    b += 6;
    R.rec_of = reinterpret_cast<uint16_t*>(b);
    return R;
}

// Bytes of dynamic LDS the record table needs; seg = 0: no tags (MODE 0).
// The tags' place also takes the list of the entry's solid slots (list_solid),
// at most `solid` of them.
__host__ __device__ inline uint32_t rec_table_bytes(uint32_t slot_words, uint32_t k, uint32_t rec_cap, uint32_t seg,
                                                    bool colors, uint32_t solid) {
    const uint32_t tags = seg ? (rec_cap / 2) * ((rec_max_kmers(slot_words, k) + seg - 1) / seg) : 0;
    return (rec_cap * slot_words + (colors ? 3 : 2) * rec_cap + 6) * 4 + (tags > solid ? tags : solid) * 2 + 4;
}

GG_DEV uint32_t rec_hash(const uint32_t* w, uint32_t sw, uint32_t color) {
    uint64_t h = 0x9E3779B97F4A7C15ULL ^ color;
    for (uint32_t i = 0; i < sw; i++) h = (h ^ w[i]) * 0xbf58476d1ce4e5b9ULL;
    h ^= h >> 31;
    return (uint32_t)h;
}

// Reverse complement of a 2-bit k-mer (k <= 32): complement every base,
// reverse the 2-bit groups.
GG_DEV uint64_t kmer_rc64(uint64_t fw, uint32_t k) {
    uint64_t x = fw ^ 0xAAAAAAAAAAAAAAAAULL;
    x = ((uint64_t)__brev((uint32_t)x) << 32) | __brev((uint32_t)(x >> 32));
    x = ((x >> 1) & 0x5555555555555555ULL) | ((x & 0x5555555555555555ULL) << 1);
    return x >> (64 - 2 * k);
}

// Canonical 2-bit k-mer (k <= 32) at base offset i of packed words (16 bases
// per word, base j at bits 2(j % 16)); *fwd when the forward strand is the
// smaller (the rolling path's fw < rc).
GG_DEV uint64_t kmer_at(const uint32_t* bw, uint32_t i, uint32_t k, bool* fwd) {
    const uint32_t wi = i >> 4, sh = (i & 15) * 2;
    const uint64_t lo = (uint64_t)bw[wi] | ((uint64_t)bw[wi + 1] << 32);
    uint64_t fw = sh ? (lo >> sh) | ((uint64_t)bw[wi + 2] << (64 - sh)) : lo;
    const uint64_t mask = (k == 32) ? ~0ULL : ((1ULL << (2 * k)) - 1);
    fw &= mask;
    const uint64_t rc = kmer_rc64(fw, k);
    *fwd = fw < rc;
    return fw < rc ? fw : rc;
}

// Both strands of the k-mer (k <= 64) at base offset i of packed words, as
// their 2-bit forms; reads the word of its first base and the three behind it.
GG_DEV void kmer_pair_at(const uint32_t* bw, uint32_t i, uint32_t k, u128_t* fw, u128_t* rc) {
    const uint32_t wi = i >> 4, sh = (i & 15) * 2;
    const u128_t w03 = (u128_t)((uint64_t)bw[wi] | ((uint64_t)bw[wi + 1] << 32)) |
                       ((u128_t)((uint64_t)bw[wi + 2] | ((uint64_t)bw[wi + 3] << 32)) << 64);
    const u128_t mask = ~(u128_t)0 >> (128 - 2 * k);
    u128_t x = w03 >> sh;
    // the fifth word is only read when the k-mer reaches into it
    if (sh + 2 * k > 128) x |= (u128_t)bw[wi + 4] << (128 - sh);
    x &= mask;
    *fw = x;
    constexpr uint64_t AA = 0xAAAAAAAAAAAAAAAAULL, M5 = 0x5555555555555555ULL;
    const uint64_t xl = (uint64_t)x ^ AA, xh = (uint64_t)(x >> 64) ^ AA;
    uint64_t l = ((uint64_t)__brev((uint32_t)xh) << 32) | __brev((uint32_t)(xh >> 32));
    uint64_t h = ((uint64_t)__brev((uint32_t)xl) << 32) | __brev((uint32_t)(xl >> 32));
    l = ((l >> 1) & M5) | ((l & M5) << 1);
    h = ((h >> 1) & M5) | ((h & M5) << 1);
    *rc = (((u128_t)h << 64) | l) >> (128 - 2 * k);
}

template <int MODE>
GG_DEV void insert_item_dedup(const MergeArgs& A, uint64_t r0, uint64_t r1, const PartWork& w, uint64_t* klo,
                              uint64_t* khi, uint32_t* st, uint32_t* vals, uint32_t* cbits, uint32_t mask, uint32_t probe_limit, uint32_t* overflow,
                              uint16_t* claimed, uint32_t* n_claimed, const RecTable& R, const uint32_t* pre,
                              uint32_t pre_color, bool hashed) {
    constexpr bool FAST = Mode<MODE>::FAST;
    constexpr uint32_t SEG = Mode<MODE>::SEG;
    const uint32_t W = Mode<MODE>::color_words(A), KW = Mode<MODE>::key_words(A);
    const uint32_t SW = Mode<MODE>::slot_words(A), k = A.k, RC = A.rec_cap;
    const uint32_t part_mask = (1u << w.log_parts) - 1;
    // one occurrence (or cnt identical ones) of a k-mer of either key width
    // returns whether it claimed table slot `at`
    auto insert_one = [&](uint64_t lo, uint64_t hi, uint32_t bits, uint32_t color, uint32_t& at) -> bool {
        uint32_t res;
        if (FAST && Mode<MODE>::TKW == 2) {
            uint64_t a, b;
            pair_of(lo, hi, a, b);
            const uint32_t h = pair_hash(a, b);
            if (part_mask && ((h >> 16) & part_mask) != w.part) return false;
            res = tab_insert_pair(klo, vals, mask, h, a, b, bits, probe_limit, at);
        } else {
            const bool one = FAST || KW == 1;
            if (part_mask) {
                const uint32_t h = one ? tab_hash64(lo) : hash128(lo, hi);
                if (((h >> 16) & part_mask) != w.part) return false;
            }
            res = one ? tab_insert64(klo, vals, mask, lo, bits, probe_limit, at)
                      : tab_insert128(klo, khi, st, vals, mask, lo, hi, bits, probe_limit, at);
        }
        if (res == 2) {
            atomicOr(overflow, 1u);
            return false;
        }
        if (W) atomicOr(&cbits[at * W + (color >> 5)], 1u << (color & 31));
        return res == 1;
    };
    auto insert_key = [&](uint64_t lo, uint64_t hi, uint32_t bits, uint32_t color) {
        if (*(volatile uint32_t*)overflow) return;
        uint32_t at = 0;
        if (insert_one(lo, hi, bits, color, at)) claimed[atomicAdd(n_claimed, 1u)] = (uint16_t)at;
    };
    // the record table's states are all free here (cleared at kernel start
    // and by phase B of the previous chunk)
    // phase A: distinct records (long records and table misses go direct);
    // thread t holds record r0 + t, loaded by the caller (pre, pre_color)
    // while the previous chunk was processed
    {
        const uint64_t r = r0 + threadIdx.x;
        if (r >= r1) goto phase_a_done;
        const uint32_t* slot = A.slots + r * SW;
        const uint32_t meta = pre[0];
        const uint32_t color = pre_color;
        bool direct = (meta & META_LONG) != 0;
        if (!direct && !hashed) {
            // the item's records are distinct: thread t's record takes the
            // first of the table slots thread t reads in phase B (t < chunk
            // <= min(rec_cap, blockDim); both powers of two)
            const uint32_t i = RC > blockDim.x ? threadIdx.x * (RC / blockDim.x) : threadIdx.x;
            for (uint32_t q = 0; q < SW; q++) R.key[i * SW + q] = pre[q];
            if (W) R.col[i] = color;
            R.cnt[i] = meta_mult(meta);
            R.state[i] = 2;
        } else if (!direct) {
            uint32_t wv[Mode<MODE>::MAX_SW];
            for (uint32_t q = 0; q < SW; q++) wv[q] = pre[q];
            uint32_t i = rec_hash(wv, SW, color) & (RC - 1);
            uint32_t probes = 0, spins = 0;
            bool done = false;
            while (!done) {
                const uint32_t sv = __hip_atomic_load(&R.state[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                if (sv == 0) {
                    if (atomicCAS(&R.state[i], 0u, 1u) == 0u) {
                        for (uint32_t q = 0; q < SW; q++) R.key[i * SW + q] = wv[q];
                        if (W) R.col[i] = color;
                        R.cnt[i] = meta_mult(meta);
                        __threadfence_block();
                        atomicExch(&R.state[i], 2u);
                        done = true;
                    }
                } else if (sv == 2) {
                    bool eq = !W || R.col[i] == color;
                    for (uint32_t q = 0; q < SW && eq; q++) eq = R.key[i * SW + q] == wv[q];
                    if (eq) {
                        atomicAdd(&R.cnt[i], meta_mult(meta));
                        done = true;
                    } else if (++probes >= 32) {
                        direct = true;
                        done = true;
                    } else {
                        i = (i + 1) & (RC - 1);
                    }
                } else if (++spins > (1u << 16)) {
                    direct = true;
                    done = true;
                }
            }
        }
        if (direct) {
            const uint32_t extra = meta_mult(meta) - 1;
            for_each_kmer<MODE>(A, slot, [&](uint64_t lo, uint64_t hi, bool is_fwd, uint32_t idx, uint32_t last) {
                insert_key(lo, hi, occurrence_bits(meta, is_fwd, idx, last) + extra, color);
            });
        }
    }
phase_a_done:
    __syncthreads();
    if (!FAST) {
        // each thread rolls the k-mers of the distinct records in its table
        // slots (rec_cap / blockDim of them) and frees the slots
        const uint32_t per = RC > blockDim.x ? RC / blockDim.x : 1u;
        const uint32_t s0 = threadIdx.x * per;
        for (uint32_t q = 0; q < per; q++) {
            const uint32_t si = s0 + q;
            if (si >= RC || R.state[si] != 2) continue;
            const uint32_t* rw = R.key + si * SW;
            const uint32_t cnt = R.cnt[si], color = W ? R.col[si] : 0u, meta = rw[0];
            for_each_kmer<MODE>(A, rw, [&](uint64_t lo, uint64_t hi, bool is_fwd, uint32_t idx, uint32_t last) {
                insert_key(lo, hi, occurrence_bits(meta, is_fwd, idx, last) - 1u + cnt, color);
            });
            R.state[si] = 0;
        }
        return;
    }
    // phase B: one exclusive scan over the table slots of their segment counts
    // places the distinct records' segments of SEG k-mers (each tagged with its
    // record's slot and its index there); each thread owns rec_cap / blockDim
    // consecutive slots (at least one) and frees them for the next chunk once
    // read.
    {
        const uint32_t per = RC > blockDim.x ? RC / blockDim.x : 1u;
        const uint32_t s0 = threadIdx.x * per;
        const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        uint32_t pk[2] = {0u, 0u};  // per <= 2 (rec_cap <= 512, 256 threads)
        uint32_t mine = 0;
        for (uint32_t q = 0; q < per; q++) {
            const uint32_t si = s0 + q;
            if (si < RC && R.state[si] == 2) {
                const uint32_t len = meta_len(R.key[si * SW]);
                const uint32_t nk = len >= k ? len - k + 1 : 0u;
                pk[q] = (nk + SEG - 1) / SEG;
                R.state[si] = 0;
            }
            mine += pk[q];
        }
        uint32_t inc = mine;
        for (uint32_t d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(inc, d);
            if (lane >= d) inc += y;
        }
        if (lane == 63) R.n[2 + wave] = inc;  // wave totals
        __syncthreads();
        uint32_t base = 0, all = 0;
        const uint32_t nw = blockDim.x >> 6;
        for (uint32_t q = 0; q < nw; q++) {
            const uint32_t t = R.n[2 + q];
            if (q < wave) base += t;
            all += t;
        }
        uint32_t run = base + inc - mine;
        for (uint32_t q = 0; q < per; q++) {
            if (pk[q]) {
                const uint32_t o = run, c = pk[q], tag = (s0 + q) << 7;
                for (uint32_t e = 0; e < c; e++) R.rec_of[o + e] = (uint16_t)(tag | e);
            }
            run += pk[q];
        }
        if (threadIdx.x == 0) R.n[1] = all;
        __syncthreads();
    }
    // phase B2: every segment of SEG k-mers of the distinct records, one per
    // thread; the first k-mer is extracted, the others rolled from it
    const uint32_t total = R.n[1];
    for (uint32_t j0 = 0; j0 < total; j0 += blockDim.x) {
        const uint32_t j = j0 + threadIdx.x;
        uint32_t cnt = 0, color = 0, meta = 0, last = 0, i0 = 0, n = 0;
        const uint32_t* bw = R.key + 1;
        if (j < total) {
            const uint32_t v = R.rec_of[j];
            const uint32_t si = v >> 7;
            i0 = (v & 127u) * SEG;
            bw = R.key + si * SW + 1;
            cnt = R.cnt[si];
            color = W ? R.col[si] : 0u;
            meta = bw[-1];
            last = meta_len(meta) - k;
            n = last + 1 - i0 < SEG ? last + 1 - i0 : SEG;
        }
        u128_t fw2 = 0, rc2 = 0;
        uint64_t fw1 = 0, rc1 = 0, next = 0;  // next: the segment's bases behind its first k-mer, 2 bits each
        if (SEG > 1 && n) {
            if (Mode<MODE>::TKW == 2) {
                kmer_pair_at(bw, i0, k, &fw2, &rc2);
            } else {
                bool fwd;
                const uint64_t c = kmer_at(bw, i0, k, &fwd);
                const uint64_t o = kmer_rc64(c, k);
                fw1 = fwd ? c : o;
                rc1 = fwd ? o : c;
            }
            const uint32_t nb = i0 + k;  // SEG - 1 <= 16 more bases: two words (the record's words end in the table)
            next = ((uint64_t)bw[nb >> 4] | ((uint64_t)bw[(nb >> 4) + 1] << 32)) >> (2 * (nb & 15));
        }
#pragma unroll
        for (uint32_t x = 0; x < SEG; x++) {
            bool cl = false;
            uint32_t at = 0;
            if (x < n) {
                uint64_t lo, hi = 0;
                bool fwd;
                if (Mode<MODE>::TKW == 2) {
                    fwd = fw2 < rc2;
                    const u128_t key = fwd ? fw2 : rc2;
                    lo = (uint64_t)key;
                    hi = (uint64_t)(key >> 64);
                } else if (SEG > 1) {
                    fwd = fw1 < rc1;
                    lo = fwd ? fw1 : rc1;
                } else {
                    lo = kmer_at(bw, i0, k, &fwd);
                }
                cl = insert_one(lo, hi, occurrence_bits(meta, fwd, i0 + x, last) - 1u + cnt, color, at);
            }
            if (SEG > 1) {
                const uint64_t c = next & 3u;
                next >>= 2;
                if (Mode<MODE>::TKW == 2) {
                    fw2 = (fw2 >> 2) | ((u128_t)c << (2 * (k - 1)));
                    rc2 = ((rc2 << 2) | (c ^ 2)) & (((u128_t)1 << (2 * k)) - 1);
                } else {
                    fw1 = (fw1 >> 2) | (c << (2 * (k - 1)));
                    rc1 = ((rc1 << 2) | (c ^ 2)) & (k == 32 ? ~0ULL : (1ULL << (2 * k)) - 1);
                }
            }
            // one LDS atomic per wavefront for the slots it claimed
            const uint64_t bal = __ballot(cl);
            if (bal) {
                const uint32_t lane = threadIdx.x & 63, first = (uint32_t)__builtin_ctzll(bal);
                uint32_t base = 0;
                if (lane == first) base = atomicAdd(n_claimed, (uint32_t)__popcll(bal));
                base = __shfl(base, (int)first);
                if (cl) claimed[base + (uint32_t)__popcll(bal & ((1ULL << lane) - 1))] = (uint16_t)at;
            }
        }
    }
}

// Work entry with the metadata a pass needs.
struct Fetched {
    uint32_t e;
    PartWork w;
    WorkItem it;  // with its slot range [it.r0, it.r1)
};

// Thread 0's pipeline of work entries: the next entry's metadata is loaded
// in two dependent steps (part entry, work item with its slot range) spread over
// the current entry's phases, and the entry after it is already claimed, so
// no barrier waits on a chain of global loads.  Entries are claimed from the
// global cursor `claim` at a time: one atomic on that single address per
// batch instead of per entry (the address serialises its atomics).
struct Pipe {
    Fetched n1;  // next entry
    uint32_t e2;  // the entry after it (claimed)
    uint32_t bat, bat_end;  // claimed batch [bat, bat_end)
};
GG_DEV uint32_t pipe_claim(const MergeArgs& A, Pipe& p) {
    if (p.bat >= p.bat_end) {
        p.bat = atomicAdd(A.work, A.claim);
        p.bat_end = p.bat + A.claim;
    }
    return p.bat < A.n_work ? p.bat++ : A.n_work;
}
GG_DEV void pipe_part(const MergeArgs& A, Pipe& p) {
    if (p.n1.e < A.n_work) p.n1.w = A.parts ? A.parts[p.n1.e] : PartWork{p.n1.e, 0u, 0u, 0u};
}
GG_DEV void pipe_item(const MergeArgs& A, Pipe& p) {
    if (p.n1.e < A.n_work) p.n1.it = A.items[p.n1.w.item];
}

// Persistent work-stealing merge: each workgroup takes work entries from a
// global cursor, thread 0 keeping the next entry's metadata in flight.
template <int MODE>
GG_DEV void merge_lds_body(const MergeArgs& A) {
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ uint32_t s_overflow;
    __shared__ Fetched s_cur;
    EmitState es{~0u, 0u};
    const uint32_t cap_max = A.lds_cap;  // the host allocates this many entries plus a margin
    // key words per table entry, then the counters; MODE 0 keeps 128-bit keys
    // in two arrays with a state word per slot behind the counters
    constexpr bool FAST = Mode<MODE>::FAST;
    const uint32_t KW = FAST ? Mode<MODE>::TKW : A.key_words;
    uint64_t* klo = reinterpret_cast<uint64_t*>(lds);
    uint64_t* khi = klo + cap_max;
    uint32_t* vals = reinterpret_cast<uint32_t*>(lds + (size_t)cap_max * 8 * KW);
    uint32_t* st = vals + cap_max;
    uint32_t* cbits = vals + (size_t)cap_max * (FAST ? 1 : KW);  // color_words per entry (colored builds)
    const uint32_t W = Mode<MODE>::color_words(A);
    uint16_t* claimed = reinterpret_cast<uint16_t*>(cbits + (size_t)cap_max * W);  // slots claimed by the entry
    __shared__ uint32_t s_solid;
    __shared__ uint32_t s_claimed;
    const bool leader = threadIdx.x == 0;
    // the table starts empty; afterwards only claimed slots are reset
    for (uint32_t i = threadIdx.x; i < cap_max; i += blockDim.x) {
        klo[i] = EMPTY64;
        if (FAST && KW == 2) klo[cap_max + i] = EMPTY64;
        vals[i] = 0;
        if (!FAST && KW == 2) st[i] = 0;
    }
    for (uint32_t i = threadIdx.x; i < cap_max * W; i += blockDim.x) cbits[i] = 0;
    if (Mode<MODE>::dedup(A)) {
        // record table slots start free; each chunk's phase B frees them again
        const RecTable R = rec_table(A, lds);
        for (uint32_t i = threadIdx.x; i < A.rec_cap; i += blockDim.x) R.state[i] = 0;
    }
    // each thread's record of the current chunk (dedup path)
    uint32_t chunk = A.rec_cap / 2;
    const uint32_t SW = Mode<MODE>::slot_words(A);
    constexpr uint32_t MSW = Mode<MODE>::MAX_SW;
    auto load_rec = [&](uint64_t r, uint64_t r_end, uint32_t* wv, uint32_t& col) {
        if (threadIdx.x < chunk && r < r_end) {
            const uint32_t* sp = A.slots + r * SW;
            // slots of 4 or 8 words, 16-byte aligned
            const uint4 v = *reinterpret_cast<const uint4*>(sp);
            wv[0] = v.x;
            wv[1] = v.y;
            wv[2] = v.z;
            wv[3] = v.w;
            if (MSW == 8 && SW == 8) {
                const uint4 u = *reinterpret_cast<const uint4*>(sp + 4);
                wv[4] = u.x;
                wv[5] = u.y;
                wv[6] = u.z;
                wv[7] = u.w;
            }
            col = W ? A.slot_color[r] : 0u;
        }
    };
    uint32_t cw[MSW] = {}, ccol = 0;
    Pipe pp{};
    if (leader) {
        s_claimed = 0;
        s_solid = 0;
        pp.bat = pp.bat_end = 0;
        pp.n1.e = pipe_claim(A, pp);
        pipe_part(A, pp);
        pipe_item(A, pp);
        pp.e2 = pp.n1.e < A.n_work ? pipe_claim(A, pp) : A.n_work;
    }
    while (true) {
        if (leader) {
            s_cur = pp.n1;
            s_overflow = 0;
            pp.n1.e = pp.e2;
            pp.e2 = (pp.e2 < A.n_work) ? pipe_claim(A, pp) : A.n_work;
            pipe_part(A, pp);
        }
        __syncthreads();
        const Fetched cur = s_cur;
        __syncthreads();
        if (cur.e >= A.n_work) break;
        const PartWork w = cur.w;
        const WorkItem it = cur.it;
        if (!A.parts && it.occ > A.lds_try) {
            if (leader) {
                A.redo[atomicAdd(A.redo_count, 1u)] = PartWork{w.item, w.part, w.log_parts, it.occ};
                pipe_item(A, pp);
            }
            continue;
        }
        uint32_t cap = 256;
        const uint64_t want = ((uint64_t)it.occ * A.table_pct + 99) / 100;
        while (cap < want && cap < cap_max) cap <<= 1;
        if (w.log_parts) cap = cap_max;
        const uint32_t mask = cap - 1;
        if (Mode<MODE>::dedup(A)) {
            const bool hashed = !A.rec_direct || it.dup;
            // records in chunks of rec_cap / 2 <= 256 (the record table's load
            // factor stays at most one half), one record per thread; identical
            // records of one chunk are counted once, the k-mer table
            // accumulates over the chunks.  Each thread's record of the next
            // chunk is loaded while the current chunk is processed.  Without
            // segment tags (MODE 0) records placed by position fill the whole
            // record table: one record per thread of the workgroup.
            chunk = (hashed || FAST) ? A.rec_cap / 2 : (A.rec_cap < blockDim.x ? A.rec_cap : blockDim.x);
            load_rec(it.r0 + threadIdx.x, it.r1, cw, ccol);
            for (uint64_t c0 = it.r0; c0 < it.r1; c0 += chunk) {
                const uint64_t c1 = c0 + chunk < it.r1 ? c0 + chunk : it.r1;
                uint32_t nw[MSW] = {}, ncol = 0;
                load_rec(c1 + threadIdx.x, it.r1, nw, ncol);
                insert_item_dedup<MODE>(A, c0, c1, w, klo, khi, st, vals, cbits, mask, 96u, &s_overflow, claimed,
                                  &s_claimed, rec_table(A, lds), cw, ccol, hashed);
#pragma unroll
                for (uint32_t q = 0; q < MSW; q++) cw[q] = nw[q];
                ccol = ncol;
                __syncthreads();  // the next chunk reuses the record table
            }
        } else {
            insert_item(A, it.r0, it.r1, w, klo, khi, st, vals, cbits, mask, 96u, &s_overflow, claimed, &s_claimed);
        }
        if (leader) pipe_item(A, pp);
        __syncthreads();
        const uint32_t n_cl = s_claimed;
        if (s_overflow) {
            // more distinct k-mers than the table holds: redone as finer parts
            if (leader) A.redo[atomicAdd(A.redo_count, 1u)] = PartWork{w.item, w.part, w.log_parts, it.occ};
        } else {
            if constexpr (Mode<MODE>::RK) {
                uint16_t* solid = rec_table(A, lds).rec_of;
                const uint32_t n = list_solid(A, vals, claimed, n_cl, solid, &s_solid);
                emit_solid<MODE>(A, it.sub, klo, khi, st, vals, cbits, solid, n, es);
            } else {
                emit_solid<MODE>(A, it.sub, klo, khi, st, vals, cbits, claimed, n_cl, es);
            }
        }
        __syncthreads();
        for (uint32_t j = threadIdx.x; j < n_cl; j += blockDim.x) {
            const uint32_t i = claimed[j];
            if (FAST && KW == 2) {
                klo[2 * i] = EMPTY64;
                klo[2 * i + 1] = EMPTY64;
            } else {
                klo[i] = EMPTY64;
            }
            vals[i] = 0;
            if (!FAST && KW == 2) st[i] = 0;
            for (uint32_t q = 0; q < W; q++) cbits[i * W + q] = 0;
        }
        if (leader) {
            s_claimed = 0;
            s_solid = 0;
        }
        __syncthreads();
    }
    close_chunk(A, es);
}

__global__ __launch_bounds__(256) void merge_lds_kernel(MergeArgs A) { merge_lds_body<0>(A); }

// The seq-hash k <= 32 variant is held to 64 VGPRs: eight waves per SIMD when
// the LDS tables allow that many workgroups.
__global__ __launch_bounds__(256, 8) void merge_lds_seq64_kernel(MergeArgs A) { merge_lds_body<1>(A); }

// The other variants: up to 128 VGPRs, for the four workgroups that a CU's LDS
// holds with their tables.
__global__ __launch_bounds__(256, 4) void merge_lds_seq64w_kernel(MergeArgs A) { merge_lds_body<2>(A); }
__global__ __launch_bounds__(256, 4) void merge_lds_rk64_kernel(MergeArgs A) { merge_lds_body<3>(A); }
__global__ __launch_bounds__(256, 4) void merge_lds_seq128_kernel(MergeArgs A) { merge_lds_body<4>(A); }
__global__ __launch_bounds__(256, 4) void merge_lds_rk128_kernel(MergeArgs A) { merge_lds_body<5>(A); }
__global__ __launch_bounds__(256, 4) void merge_lds_col64_kernel(MergeArgs A) { merge_lds_body<6>(A); }
__global__ __launch_bounds__(256, 4) void merge_lds_col128_kernel(MergeArgs A) { merge_lds_body<7>(A); }

// Makes the solid table dense: with T = off[n_chunks] entries in all (off: the
// exclusive scan of the chunks' fill counts), the entries at positions >= T
// move, in order, into the free positions below T, which are as many.  Every
// wavefront of the merge leaves its last chunk partly filled, so a table of T
// entries used to span T plus about 2048 positions per wavefront (35 K entries
// of a 30 kbp genome: 16 M positions), all of which the copy to the host, the
// query index and the unitigs had to visit, chunk by chunk.  One workgroup per
// chunk; at most min(T, free positions) entries move (each read and written
// once), a thread finding its destination by a binary search over the chunks'
// free-position counts.  Bound by HBM: 0.1 ms beside a 10.9 ms merge on 57.7 M
// entries.  Measured with the table's consumers: build and copy of 36 K entries
// to the host 60.2 -> 0.9 ms, of 0.83 M entries 83.7 -> 3.0 ms; unitigs of
// 0.84 M entries with 128-bit keys 5.8 -> 2.6 ms.
__global__ __launch_bounds__(256) void out_close_holes_kernel(const uint64_t* off, uint32_t n_chunks, uint64_t* key,
                                                              uint32_t key_words, uint32_t* val, uint32_t* sub,
                                                              uint32_t* colors, uint32_t color_words) {
    const uint64_t T = off[n_chunks];
    const uint32_t ct = (uint32_t)(T / OUT_CHUNK);  // the chunk holding position T (n_chunks when all are full)
    const uint32_t c = blockIdx.x;
    if (c < ct) return;
    const uint32_t limit = (uint32_t)(T - (uint64_t)ct * OUT_CHUNK);  // positions of chunk ct below T
    const uint32_t fill_t = ct < n_chunks ? (uint32_t)(off[ct + 1] - off[ct]) : 0u;
    const uint32_t first = c == ct ? (fill_t < limit ? fill_t : limit) : 0u;  // entries of this chunk that stay
    const uint32_t fill = (uint32_t)(off[c + 1] - off[c]);
    // entries at positions >= T before this chunk
    const uint64_t moved = c == ct ? 0 : off[c] - off[ct] - (fill_t < limit ? fill_t : limit);
    for (uint32_t i = first + threadIdx.x; i < fill; i += blockDim.x) {
        const uint64_t r = moved + (i - first);
        // the chunk h <= ct with the r-th free position: the last one with at
        // most r free positions before it
        uint32_t lo = 0, hi = ct;
        while (lo < hi) {
            const uint32_t mid = (lo + hi + 1) >> 1;
            if ((uint64_t)mid * OUT_CHUNK - off[mid] <= r) lo = mid; else hi = mid - 1;
        }
        const uint64_t src = (uint64_t)c * OUT_CHUNK + i;
        const uint64_t dst = (uint64_t)lo * OUT_CHUNK + (off[lo + 1] - off[lo]) + (r - ((uint64_t)lo * OUT_CHUNK - off[lo]));
        for (uint32_t q = 0; q < key_words; q++) key[dst * key_words + q] = key[src * key_words + q];
        val[dst] = val[src];
        sub[dst] = sub[src];
        for (uint32_t q = 0; q < color_words; q++) colors[dst * color_words + q] = colors[src * color_words + q];
    }
}

// The two halves of cross-unit boundary k-mers (the fixup list's n entries)
// combined and put behind the table's T entries: a wavefront per entry compares
// it with all others, 64 at a time, and the first of a key takes the flags and
// colors of the rest.  n^2 comparisons of cached reads: below FIX_JOIN_MAX
// entries that beats copying the list out and back (eight copies), above it the
// host sorts the list.  With a thread per entry and a pass over the list per
// color word the merge of 300 colors (16 MB, 844 entries) took 4.7 ms, 3.5 now,
// of 1000 colors (52 MB, 2262 entries) 38.6, 30.8 now.
constexpr uint32_t FIX_JOIN_MAX = 4096;
__global__ __launch_bounds__(256) void fix_join_kernel(const uint64_t* fk, const uint32_t* fv, const uint32_t* fs,
                                                       const uint32_t* fc, uint32_t n, uint32_t key_words,
                                                       uint32_t color_words, const uint64_t* table_end, uint64_t cap,
                                                       uint64_t* key, uint32_t* val, uint32_t* sub, uint32_t* colors,
                                                       unsigned long long* added) {
    const uint32_t i = (blockIdx.x * blockDim.x + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (i >= n) return;
    const uint32_t s = fs[i];
    const uint64_t lo = fk[(uint64_t)i * key_words], hi = key_words == 2 ? fk[2 * (uint64_t)i + 1] : 0;
    uint32_t flags = 0, bits = 0;  // bits: color word `lane` (a build has at most 32)
    for (uint32_t j0 = 0; j0 < n; j0 += 64) {
        const uint32_t j = j0 + lane;
        const bool same = j < n && fs[j] == s && fk[(uint64_t)j * key_words] == lo &&
                          (key_words == 1 || fk[2 * (uint64_t)j + 1] == hi);
        uint64_t m = __ballot(same);
        // entries before i come in earlier steps or lower lanes
        if (m && j0 + (uint32_t)__builtin_ctzll(m) < i) return;
        if (same) flags |= fv[j];
        if (lane < color_words)
            for (; m; m &= m - 1) bits |= fc[(uint64_t)(j0 + (uint32_t)__builtin_ctzll(m)) * color_words + lane];
    }
    const uint32_t both = (__ballot(flags >> 31) ? 1u << 31 : 0u) | (__ballot((flags >> 30) & 1u) ? 1u << 30 : 0u);
    unsigned long long pos = 0;
    if (lane == 0) pos = *table_end + atomicAdd(added, 1ULL);
    pos = __shfl(pos, 0);
    if (pos >= cap) return;  // the host sees the count and retries with more room
    if (lane == 0) {
        key[pos * key_words] = lo;
        if (key_words == 2) key[2 * pos + 1] = hi;
        val[pos] = fv[i] | both;
        sub[pos] = s;
    }
    if (lane < color_words) colors[pos * color_words + lane] = bits;
}

// Entry values split into multiplicities and flags for a copy to the host.
__global__ void out_split_kernel(const uint32_t* val, uint64_t n, uint32_t* mult, uint8_t* flags) {
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t v = val[i];
        mult[i] = v & 0x3FFFFFFFu;
        flags[i] = (uint8_t)(v >> 30);
    }
}

// One thread per sub-bucket: runs of its units become work items of at most
// `group_occ` occurrences (a single unit above that is an item of its own),
// each with its slot range.  An item is marked dup when one of its units
// stores more than `dd_max` records: the compaction deduplicates units of up
// to dd_max records, so only such units can still hold identical records.
__global__ void make_items_kernel(const uint32_t* unit_kmers, const uint64_t* unit_off, uint32_t n_sub, uint32_t xb,
                                  uint32_t group_occ, uint32_t dd_max, WorkItem* items, unsigned int* n_items) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n_sub) return;
    const uint32_t u_begin = s << xb, u_end = (s + 1) << xb;
    uint32_t start = u_begin, acc = 0, dup = 0;
    for (uint32_t u = u_begin; u < u_end; u++) {
        const uint32_t o = unit_kmers[u];
        if (acc == 0 && o == 0) {
            start = u + 1;
            continue;
        }
        if (acc > 0 && acc + o > group_occ) {
            items[atomicAdd(n_items, 1u)] = WorkItem{start, dup, acc, s, unit_off[start], unit_off[u]};
            start = u;
            acc = 0;
            dup = 0;
        }
        acc += o;
        if (unit_off[u + 1] - unit_off[u] > dd_max) dup = 1;
    }
    if (acc > 0) items[atomicAdd(n_items, 1u)] = WorkItem{start, dup, acc, s, unit_off[start], unit_off[u_end]};
}

}  // namespace gg
