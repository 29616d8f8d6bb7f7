// unitigs.hip -- in/out extension flags and intra-sub-bucket unitig chains
// over the solid seq-hash table of the last merge.
//
// Restates the extension of crates/assembler_kmers_merge/src/unitigs_extender/
// hashmap.rs:162-297,442-601 as an order-free rule (the reference's greedy
// loop gives the same chains except where a k-mer's flagged side has a
// neighbour in its own sub-bucket, where its own result depends on the order
// in which it visits k-mers):
//   * in a k-mer's canonical orientation, side 0 is the predecessor side and
//     side 1 the successor side; its degree on a side is the number of solid
//     k-mers of the same sub-bucket one base away (manual_roll_forward /
//     manual_roll_reverse, crates/hashes/src/base/cn_seqhash_base.rs:165-200);
//   * a k-mer whose flags are exactly INCL_BEGIN (or INCL_END) has its side 0
//     (or side 1) flagged: its continuation is in another bucket
//     (contig_break, hashmap.rs:287-292; begin/end_ignored, :483-494);
//   * sides (p,s) and (q,t) are linked when each is the other's only
//     neighbour, p != q, and neither side is flagged;
//   * a unitig is a maximal linked path, written from its end with the
//     smaller (key, side); an end is open when its outer side is flagged.
// Cycles (paths without ends) are rare and are walked on the host.
//
// Joined mode (global != 0) builds the maximal unitigs of the whole solid
// set, i.e. the partial unitigs of every sub-bucket joined across buckets
// (what the links / reorganize / build_final_unitigs stages of
// crates/assembler_pipeline/src/extend_unitigs.rs:348-993 produce): a k-mer
// held by several sub-buckets (a boundary k-mer, counted on both sides) is
// one node, represented by its smallest table position; neighbours are
// looked up over the whole table and no side is flagged.
#include "common.h"

namespace gg {

constexpr uint32_t NO_LINK = 0xFFFFFFFFu;

struct UnitigArgs {
    const uint64_t* out_key;
    const uint32_t* out_val;
    const uint32_t* out_sub;
    uint32_t key_words;
    uint32_t k;
    uint64_t* tab;  // [tab_mask + 1] open addressing: hash bits 32-63 << 32 | (position + 1); 0 = empty
    uint64_t tab_mask;
    uint32_t* nb;  // [2 n_pos] only neighbour (q << 1 | t) or NO_LINK
    uint8_t* ext;  // [n_pos] degree side 0 (0, 1, 2 = more) | degree side 1 << 2
    uint32_t* link;  // [2 n_pos]
    uint64_t* seg;  // [2 groups of SPLIT positions] rest of the path behind each splitter, see seg_pair
    uint64_t* head;  // [2 n_pos] the same for path ends (other entries unused)
    uint32_t* uni_of;  // [2 n_pos] unitig written from this end, NO_LINK when written from its other end
    uint32_t* uni_bytes;  // [unitigs]
    const uint64_t* uni_off;  // [unitigs + 1] exclusive scan of uni_bytes
    unsigned long long* totals;  // unitigs, bytes, duplicate entries (joined mode)
    uint8_t* seq;
    uint32_t* uni_sub;
    uint8_t* uni_flags;
    uint8_t* visited;  // [n_pos]
    uint32_t global;  // joined mode: one graph over all sub-buckets
    uint8_t* rep;  // [n_pos] joined mode: 1 where p is its key's smallest position
    uint32_t mark_visited;  // write pass: mark path nodes (needed only when cycles exist)
    uint32_t* path_pos;  // write pass, optional: the table position of every k-mer of every unitig, in
                         // written order (unitig i's k-mers start at uni_off[i] - i * k)
};

// Position p is a node of the graph being compacted.
GG_DEV bool unitig_valid(const UnitigArgs& A, uint64_t p) { return !A.global || A.rep[p]; }

GG_DEV u128_t key_at(const UnitigArgs& A, uint64_t p) {
    const uint64_t lo = A.out_key[p * A.key_words];
    const uint64_t hi = A.key_words == 2 ? A.out_key[p * 2 + 1] : 0;
    return ((u128_t)hi << 64) | lo;
}

// Reverse complement of a k-mer (base j at bits 2j, A0 C1 T2 G3, so the
// complement of a base is code ^ 2): complement all 64 positions, reverse
// the 128 bits, swap the bits inside each 2-bit group back, and drop the
// 64 - k positions above the k-mer, which the reversal put at the bottom.
GG_DEV u128_t kmer_rc128(u128_t x, uint32_t k) {
    constexpr uint64_t AA = 0xAAAAAAAAAAAAAAAAULL, M5 = 0x5555555555555555ULL;
    uint64_t lo = __brevll((uint64_t)(x >> 64) ^ AA), hi = __brevll((uint64_t)x ^ AA);
    lo = ((lo >> 1) & M5) | ((lo & M5) << 1);
    hi = ((hi >> 1) & M5) | ((hi & M5) << 1);
    const u128_t r = ((u128_t)hi << 64) | lo;
    return r >> (128 - 2 * k);
}

GG_DEV bool side_flagged(const UnitigArgs& A, uint64_t p, uint32_t s) {
    if (A.global) return false;
    const uint32_t fl = A.out_val[p] >> 30;
    return (fl == 1 && s == 0) || (fl == 2 && s == 1);
}

// Every position goes into the lookup table (linear probing; the table has at
// least twice as many slots as positions, so probing ends).  In joined mode a
// key's second entry is found here: the slot keeps the smaller position, the
// other one stops being a representative (rep starts at 1 everywhere) and is
// counted, so each key has one slot and a lookup ends at its first match.
__global__ __launch_bounds__(256) void utab_insert_kernel(UnitigArgs A, uint64_t n_pos) {
    __shared__ unsigned int part[4];
    unsigned int dup = 0;
    for (uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; p < n_pos;
         p += (uint64_t)gridDim.x * blockDim.x) {
        const u128_t c = key_at(A, p);
        const uint64_t h = index_hash((uint64_t)c, (uint64_t)(c >> 64));
        const unsigned long long v = (h & 0xFFFFFFFF00000000ULL) | (p + 1);
        for (uint64_t i = h & A.tab_mask;; i = (i + 1) & A.tab_mask) {
            unsigned long long* slot = reinterpret_cast<unsigned long long*>(A.tab + i);
            const unsigned long long cur = atomicCAS(slot, 0ULL, v);
            if (cur == 0ULL) break;
            // a slot's key never changes, only which of its positions it names
            if (A.global && (uint32_t)(cur >> 32) == (uint32_t)(v >> 32) && key_at(A, (uint32_t)cur - 1u) == c) {
                const unsigned long long old = atomicMin(slot, v);
                A.rep[old > v ? (uint32_t)old - 1u : (uint32_t)p] = 0;
                dup++;
                break;
            }
        }
    }
    if (!A.global) return;
    for (uint32_t d = 32; d; d >>= 1) dup += __shfl_down(dup, d);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = dup;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned int t = part[0] + part[1] + part[2] + part[3];
        if (t) atomicAdd(A.totals + 2, (unsigned long long)t);
    }
}

// Position of key `c` inside sub-bucket `sub`, or NO_LINK.  In joined mode
// the sub-bucket is ignored and the key's representative is returned.
GG_DEV uint32_t lookup_in_sub(const UnitigArgs& A, u128_t c, uint32_t sub) {
    const uint64_t h = index_hash((uint64_t)c, (uint64_t)(c >> 64));
    const uint32_t fp = (uint32_t)(h >> 32);
    for (uint64_t i = h & A.tab_mask;; i = (i + 1) & A.tab_mask) {
        const uint64_t v = A.tab[i];
        if (v == 0) return NO_LINK;
        if ((uint32_t)(v >> 32) != fp) continue;
        const uint32_t q = (uint32_t)v - 1u;
        if (key_at(A, q) == c && (A.global || A.out_sub[q] == sub)) return q;
    }
}

__global__ void ext_kernel(UnitigArgs A, uint64_t n_pos) {
    const uint32_t k = A.k;
    const u128_t mask = (k >= 64) ? ~(u128_t)0 : (((u128_t)1 << (2 * k)) - 1);
    for (uint64_t p = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; p < n_pos; p += (uint64_t)gridDim.x * blockDim.x) {
        if (!unitig_valid(A, p)) {
            A.nb[2 * p] = A.nb[2 * p + 1] = NO_LINK;
            A.ext[p] = 0;
            continue;
        }
        const u128_t x = key_at(A, p);
        const u128_t xr = kmer_rc128(x, k);
        const uint32_t sub = A.out_sub[p];
        uint32_t degs = 0;
        for (uint32_t s = 0; s < 2; s++) {
            uint32_t cnt = 0, only = NO_LINK;
            for (uint32_t b = 0; b < 4; b++) {
                // neighbour y and its reverse complement, both from x and rc(x)
                const u128_t y = s ? ((x >> 2) | ((u128_t)b << (2 * (k - 1)))) : (((x << 2) | b) & mask);
                const u128_t yr = s ? (((xr << 2) | (b ^ 2u)) & mask) : ((xr >> 2) | ((u128_t)(b ^ 2u) << (2 * (k - 1))));
                const u128_t c = y < yr ? y : yr;
                const uint32_t q = lookup_in_sub(A, c, sub);
                if (q == NO_LINK) continue;
                cnt++;
                const uint32_t t = (y == c) ? (s ? 0u : 1u) : (s ? 1u : 0u);
                only = (q << 1) | t;
            }
            A.nb[2 * p + s] = cnt == 1 ? only : NO_LINK;
            degs |= (cnt > 2 ? 2u : cnt) << (2 * s);
        }
        A.ext[p] = (uint8_t)degs;
    }
}

__global__ void link_kernel(UnitigArgs A, uint64_t n_pos) {
    for (uint64_t e = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; e < 2 * n_pos;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t v = A.nb[e];
        uint32_t out = NO_LINK;
        if (v != NO_LINK) {
            const uint64_t p = e >> 1, q = v >> 1;
            const uint32_t s = (uint32_t)(e & 1), t = v & 1;
            if (q != p && !side_flagged(A, p, s) && !side_flagged(A, q, t) && A.nb[v] == (uint32_t)e) out = v;
        }
        A.link[e] = out;
    }
}

// Last base of k-mer q read in orientation t (0: canonical, 1: reverse
// complement): base k-1 of the key, or the complement of its base 0.
GG_DEV uint32_t entry_base(const UnitigArgs& A, uint64_t q, uint32_t t) {
    if (t) return ((uint32_t)A.out_key[q * A.key_words] & 3u) ^ 2u;
    const uint32_t j = A.k - 1;
    const uint64_t w = A.out_key[q * A.key_words + (j >> 5)];
    return (uint32_t)(w >> (2 * (j & 31))) & 3u;
}

// Writes the bytes of one unitig at seq[off...] through 4-byte stores; the
// first and last words, which it may share with its neighbours, byte by byte.
struct SeqWriter {
    uint8_t* seq;
    uint64_t off, a;
    uint32_t acc = 0;
    GG_DEV SeqWriter(uint8_t* s, uint64_t o) : seq(s), off(o), a(o) {}
    GG_DEV void put(uint32_t ch) {
        acc |= ch << (8 * (uint32_t)(a & 3));
        if ((a & 3) == 3) {
            if (a - 3 >= off) {
                *reinterpret_cast<uint32_t*>(seq + a - 3) = acc;
            } else {
                for (uint64_t b = off; b <= a; b++) seq[b] = (uint8_t)(acc >> (8 * (uint32_t)(b & 3)));
            }
            acc = 0;
        }
        a++;
    }
    GG_DEV void finish() {
        if ((a & 3) == 0) return;  // the last word was stored
        const uint64_t w0 = a & ~(uint64_t)3;
        for (uint64_t b = w0 > off ? w0 : off; b < a; b++) seq[b] = (uint8_t)(acc >> (8 * (uint32_t)(b & 3)));
    }
};

// ---- paths ------------------------------------------------------------------
// A path is walked along directed elements e = 2 p + side entered; the next one
// is link[e ^ 1].  Walking a whole path by one thread costs its length times
// the latency of a dependent read (one error-free genome is one path), so paths
// are cut at splitters: one position in each group of SPLIT, chosen by a hash.
// Every splitter and every path end walks to the next splitter (SPLIT nodes on
// average), splitters then jump over each other (pointer doubling on 1 / SPLIT
// of the nodes), after which every end knows its path's length and other end,
// and the segments write their part of the unitig, all at once.
// 14.4 M entries, joined: lengths and ends 1.5 -> 1.2 ms, writing 2.9 -> 2.0 ms
// (now bound by a random link and key read per node); one path of 400 K nodes
// no longer sets the time.
constexpr uint32_t SPLIT = 16;

GG_DEV uint64_t split_pos(uint64_t group) { return group * SPLIT + (mix64(group) & (SPLIT - 1)); }
GG_DEV bool is_split(uint64_t p) { return split_pos(p / SPLIT) == p; }

// From an element: nodes up to `to` (exclusive of it while not done), and
// whether the path ends there: `to` is then the path's last element, else the
// next splitter's.
constexpr uint32_t SEG_DONE = 1u << 31;
GG_DEV uint64_t seg_pair(uint32_t nodes, bool done, uint32_t to) {
    return ((uint64_t)(nodes | (done ? SEG_DONE : 0u)) << 32) | to;
}
GG_DEV bool seg_done(uint64_t x) { return (x >> 63) != 0; }
GG_DEV uint32_t seg_nodes(uint64_t x) { return (uint32_t)(x >> 32) & ~SEG_DONE; }
// x followed by y, the pair of the element x leads to (cycles never end: their
// count wraps inside its 31 bits and is not used)
GG_DEV uint64_t seg_join(uint64_t x, uint64_t y) {
    return seg_pair((seg_nodes(x) + seg_nodes(y)) & ~SEG_DONE, seg_done(y), (uint32_t)y);
}
GG_DEV uint64_t* seg_of(const UnitigArgs& A, uint64_t e) { return A.seg + 2 * ((e >> 1) / SPLIT) + (e & 1); }

// Every splitter and path end to the next splitter or the path's end.
__global__ void seg_walk_kernel(UnitigArgs A, uint64_t n_pos) {
    for (uint64_t e = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; e < 2 * n_pos;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const bool split = is_split(e >> 1), head = A.link[e] == NO_LINK;
        if ((!split && !head) || !unitig_valid(A, e >> 1)) continue;
        uint64_t cur = e, x = 0;
        for (uint32_t nodes = 1;; nodes++) {
            const uint32_t nx = A.link[cur ^ 1];
            if (nx == NO_LINK || is_split(nx >> 1)) {
                x = seg_pair(nodes, nx == NO_LINK, nx == NO_LINK ? (uint32_t)cur : nx);
                break;
            }
            cur = nx;
        }
        if (split) *seg_of(A, e) = x;
        if (head) A.head[e] = x;
    }
}

// One round: every splitter's pair joined with those of the splitters it leads
// to, up to SEG_HOPS times.  In place: a pair is one 8-byte word, and whatever
// round's pair is read leads as far as it says.
constexpr uint32_t SEG_HOPS = 8;
__global__ void seg_jump_kernel(UnitigArgs A, uint64_t n_pos) {
    const uint64_t n = 2 * ((n_pos + SPLIT - 1) / SPLIT);
    for (uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t p = split_pos(i >> 1);
        if (p >= n_pos || !unitig_valid(A, p)) continue;
        uint64_t x = A.seg[i];
        if (seg_done(x)) continue;
        for (uint32_t h = 0; h < SEG_HOPS && !seg_done(x); h++)
            x = seg_join(x, __hip_atomic_load(seg_of(A, (uint32_t)x), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
        atomicExch(reinterpret_cast<unsigned long long*>(A.seg + i), (unsigned long long)x);
    }
}

// Path ends: the end with the smaller (key, side) becomes the head of a unitig
// (listed in arrival order, with its bytes: k-mer, one base per further k-mer,
// '\n').  Each thread takes two positions; one atomic per workgroup and step.
__global__ __launch_bounds__(256) void head_kernel(UnitigArgs A, uint64_t n_pos) {
    __shared__ uint32_t wave_n[4];
    __shared__ uint32_t s_base;
    __shared__ unsigned long long s_bytes[4];
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, k = A.k;
    const uint64_t ne = 2 * n_pos, step = (uint64_t)gridDim.x * 1024;
    unsigned long long bytes = 0;
    for (uint64_t e0 = (uint64_t)blockIdx.x * 1024; e0 < ne; e0 += step) {
        uint32_t len[4], n = 0;
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            const uint64_t e = e0 + 4 * threadIdx.x + j;
            len[j] = 0;
            if (e >= ne || A.link[e] != NO_LINK || !unitig_valid(A, e >> 1)) continue;
            uint64_t x = A.head[e];
            if (!seg_done(x)) x = seg_join(x, *seg_of(A, (uint32_t)x));
            A.head[e] = x;
            const uint64_t p = e >> 1, last = (uint32_t)x, q = last >> 1;
            const u128_t kp = key_at(A, p), kq = key_at(A, q);
            const bool canon = kp < kq || (kp == kq && (uint32_t)(e & 1) < (uint32_t)((last ^ 1) & 1));
            if (canon) {
                len[j] = seg_nodes(x) + k;
                bytes += len[j];
                n++;
            } else {
                A.uni_of[e] = NO_LINK;
            }
        }
        uint32_t inc = n;
        for (uint32_t d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(inc, d);
            if (lane >= d) inc += y;
        }
        if (lane == 63) wave_n[wave] = inc;
        __syncthreads();
        uint32_t before = 0, all = 0;
        for (uint32_t w = 0; w < 4; w++) {
            if (w < wave) before += wave_n[w];
            all += wave_n[w];
        }
        if (threadIdx.x == 0) s_base = all ? (uint32_t)atomicAdd(A.totals, (unsigned long long)all) : 0u;
        __syncthreads();
        uint32_t i = s_base + before + inc - n;
#pragma unroll
        for (uint32_t j = 0; j < 4; j++) {
            if (!len[j]) continue;
            const uint64_t e = e0 + 4 * threadIdx.x + j;
            A.uni_bytes[i] = len[j];
            A.uni_of[e] = i++;
        }
        __syncthreads();  // wave_n and s_base are reused
    }
    for (uint32_t d = 32; d; d >>= 1) bytes += __shfl_down(bytes, d);
    if (lane == 0) s_bytes[wave] = bytes;
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long t = s_bytes[0] + s_bytes[1] + s_bytes[2] + s_bytes[3];
        if (t) atomicAdd(A.totals + 1, t);
    }
}

// Every segment of a unitig writes its bases (its first node's place is the
// path's length less what is left of it), the head's segment the first k-mer,
// the last one the '\n'; segments against the unitig's direction write nothing.
__global__ void seg_write_kernel(UnitigArgs A, uint64_t n_pos) {
    const uint32_t k = A.k;
    constexpr uint32_t ASCII = 'A' | ('C' << 8) | ('T' << 16) | ('G' << 24);
    for (uint64_t e = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; e < 2 * n_pos;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint64_t p = e >> 1;
        const uint32_t s = (uint32_t)(e & 1);
        const bool is_head = A.link[e] == NO_LINK;
        if ((!is_head && !is_split(p)) || !unitig_valid(A, p)) continue;
        const uint64_t x = is_head ? A.head[e] : *seg_of(A, e);
        if (!seg_done(x)) continue;  // on a cycle
        // the path's last element entered from behind is the end of the
        // opposite direction, whose last element is this direction's head
        const uint32_t h = is_head ? (uint32_t)e : (uint32_t)A.head[(uint32_t)x ^ 1u] ^ 1u;
        const uint32_t ui = A.uni_of[h];
        if (ui == NO_LINK) continue;
        const uint64_t off = A.uni_off[ui];
        uint32_t j = seg_nodes(A.head[h]) - seg_nodes(x);  // index of node p in the path
        SeqWriter out(A.seq, j ? off + k - 1 + j : off);
        if (j == 0) {
            const u128_t y = s == 0 ? key_at(A, p) : kmer_rc128(key_at(A, p), k);
            for (uint32_t i = 0; i < k; i++) out.put((ASCII >> (8 * ((uint32_t)(y >> (2 * i)) & 3u))) & 0xFFu);
            A.uni_sub[ui] = A.global ? 0u : A.out_sub[p];
            const uint64_t last = (uint32_t)x;
            A.uni_flags[ui] = (uint8_t)((side_flagged(A, p, s) ? 1u : 0u) |
                                        (side_flagged(A, last >> 1, (uint32_t)((last ^ 1) & 1)) ? 2u : 0u));
        } else {
            out.put((ASCII >> (8 * entry_base(A, p, s))) & 0xFFu);
        }
        uint32_t* pp = A.path_pos ? A.path_pos + (off - (uint64_t)ui * k) : nullptr;
        uint64_t cur = e;
        while (true) {
            const uint64_t q = cur >> 1;
            if (A.mark_visited) A.visited[q] = 1;
            if (pp) pp[j++] = (uint32_t)q;
            const uint32_t nx = A.link[cur ^ 1];
            if (nx == NO_LINK) {
                out.put('\n');
                break;
            }
            if (is_split(nx >> 1)) break;
            cur = nx;
            out.put((ASCII >> (8 * entry_base(A, cur >> 1, (uint32_t)(cur & 1)))) & 0xFFu);
        }
        out.finish();
    }
}

}  // namespace gg
