// bucketing.hip -- minimizer bucketing on gfx950.
//
// Restates, for the device, the per-run work of
//   crates/assembler_minimizer_bucketing/src/lib.rs:171-270  (process_sequence)
//   crates/hashes/src/cn_nthash.rs:19-109                     (canonical ntHash m-mers)
//   crates/hashes/src/rolling/batch_minqueue.rs:37-189        (window minima + splits)
//   crates/minimizer_bucketing/src/sequences_splitter.rs:15-40 (runs of >= k ACGT)
//
// Input layout: one byte array in HBM holding every record followed by a
// separator byte.  Any byte that is not A/C/G/T (either case) ends an ACGT run,
// exactly like 'N' after the reference's normalisation, so separators need no
// index.
//
// Geometry.  A "window" j is the (k-1)-mer starting at base j; its minimum is
// taken over the w = k - m m-mers j .. j+w-1.  A tile owns windows [t0, t0+T)
// and is processed by one wavefront.  The wave also computes the w windows
// before t0 (halo), enough to find the start of every group whose minimizer is
// unique (such groups span at most w windows).  Groups with a non-unique
// minimizer may be longer; their start is found in the global group-start
// bitmap once pass 1 has written all of it.
//
//   pass 1 (bucket_stage_kernel)  : group-start bitmap; every record built,
//                                   counted in its unit (the count is its rank)
//                                   and written to its unit's region at that
//                                   rank, or to the spill list past the region
//          (bucket_defer_kernel)  : records whose group starts before the halo
//   scan   (scan_*_kernel)        : unit offsets of the dense arena
//   pass 2 (unit_compact_kernel)  : each unit's region copied to its offsets
//          (spill_place_kernel)   : spilled records to unit offset + rank
//
// A group = maximal run of consecutive windows sharing the minimizer (value,
// and position when unique).  Its super-k-mer is the set of k-mers touching
// the group: bases [a-1, b+k) for a group of windows [a, b], clipped to the
// ACGT run (include_first / include_last when clipped).
#include "common.h"

namespace gg {

// 64-bit words of the rolling-hash tables (BucketArgs::gtab).
constexpr uint32_t GTAB_WORDS = 2 * (20 + 16);

// Stripes of the spill list, their cursors a line apart: the updates of one
// cursor wait for each other (0.23 Gbases with m = 11, whose frequent minimizers
// overfill 3 % of the units: staging pass 2.4 ms with one, 1.4 to 1.8 with 64).
constexpr uint32_t SPILL_STRIPES = 64;
constexpr uint32_t SPILL_STRIDE = 8;

// Records are scattered by physical unit: the sub-bucket (the semantic unit,
// one kmers_transform job) refined by `xb` further bits of the minimizer hash
// for unique minimizers.  Units of one sub-bucket are contiguous, so the merge
// can process any run of them as one work item.
struct BucketArgs {
    const uint8_t* seq;
    uint64_t n;  // bytes in seq
    uint32_t k, m, w;
    uint32_t b, sb, xb;
    uint32_t canonical;
    uint32_t T;  // windows per tile (multiple of 32)
    uint64_t n_tiles;
    uint64_t tile0;  // index of the launch's first tile (launches over part of the tiles)
    uint32_t* seg_bits;  // [ceil(n/32)+2] group-start bitmap (written by pass 1)
    uint32_t* sub_count;  // [n_units] records per unit
    unsigned long long* unit_ck;  // [n_units] records << 32 | k-mer occurrences, counted in pass 1
    uint64_t n_slots;  // slots in the arena
    // Pass 1 writes record `rank` of unit u to its region slot
    // u * unit_cap + rank; records of rank >= unit_cap are appended to the
    // spill list with their unit and rank.
    uint32_t unit_cap;
    uint32_t* region;  // [n_units * unit_cap * slot_words]
    uint32_t* region_color;  // [n_units * unit_cap] (colored builds)
    // the list is cut into spill_stripes (a power of two, at most SPILL_STRIPES)
    // of spill_cap entries, a workgroup appending to the one of its index
    uint32_t* spill_slots;  // [spill_stripes * spill_cap * slot_words]
    uint32_t* spill_unit;  // [spill_stripes * spill_cap]
    uint32_t* spill_rank;  // [spill_stripes * spill_cap]
    uint32_t* spill_color;  // [spill_stripes * spill_cap] (colored builds)
    unsigned long long* spill_cursor;  // a stripe's records at SPILL_STRIDE * stripe (may exceed spill_cap: the host retries)
    uint64_t spill_cap;
    uint32_t spill_stripes;
    uint64_t* defer;  // [n_tiles * 3] records whose group starts before the tile: end window, minimizer, last flag
    unsigned int* defer_count;
    unsigned long long* kmer_total;  // k-mer occurrences of all records
    const uint64_t* sub_off;  // [n_units+1] slot offsets
    uint32_t* slots;
    uint32_t slot_words;
    uint32_t* pool;
    unsigned long long* pool_cursor;
    uint64_t pool_cap;  // words
    uint32_t* sub_kmers;  // [n_units] k-mer occurrences
    // after deduplication: records stored per unit (distinct region records
    // plus spilled ones), of which distinct region records
    uint32_t* unit_dcount;
    uint32_t* unit_dregion;
    // k-mer positions per unit once identical records are stored once (the
    // inserts the merge makes; sizes its work items and tables)
    uint32_t* unit_skmers;
    const uint64_t* color_starts;
    const uint32_t* colors;
    uint32_t n_colors;
    uint32_t* slot_color;
    uint32_t* error_flag;  // set when a consistency check fails
    // interleaved (fw, rc) rolling tables: entries 0..19 index out*4+in, then
    // two bases c0 | c1 << 2 that come in while none leaves
    uint64_t gtab[GTAB_WORDS];
};

// m-mers of one tile: 16 per lane of its wavefront.
constexpr uint32_t TILE_MMERS = 1024;

// Windows computed before a tile's own ones: at least w (a unique minimizer's
// group spans at most w windows), a multiple of the lanes' 16.
__host__ __device__ inline uint32_t tile_halo(uint32_t w) { return (w + 15) / 16 * 16; }

// Windows per tile: the tile's windows, its halo and the window behind them
// take m-mers 0 .. halo + T + w - 1; whole 32-bit words of the bitmap.
__host__ __device__ inline uint32_t tile_windows(uint32_t w) { return (TILE_MMERS - tile_halo(w) - w) / 32 * 32; }

// Block of the window minima (see tile_minima): the largest power of two that
// is at most min(w, 16).
__host__ __device__ inline uint32_t tile_block(uint32_t w) { return w >= 16 ? 16 : w >= 8 ? 8 : w >= 4 ? 4 : 2; }

// The w == 16 variant: its invalid-base slice of 64 bits covers the windows of
// a lane for k <= 47.
__host__ __device__ inline bool tile_w16(uint32_t w, uint32_t k) { return w == 16 && k <= 47; }

// LDS of a workgroup of that variant, with the kernel's own 2064 bytes 9
// allocation units of 1280: a CU holds 14 wavefronts where its tile alone allows
// 16.  The records' atomics and stores run at 20 G/s each while few enough
// wavefronts wait in them and at 12 G/s once too many do (the L2s' write requests
// to memory then stall, 69 M stall cycles against 1 M), and how many that is
// depends on where the buffers lie in memory, which changes with what was
// allocated before.  Cheaper hashes or input bytes bring wavefronts there sooner,
// so neither helps.  Staging pass where few are too many and where 16 are not:
//   bytes four at a time, 16 wavefronts: 1 Gbase 9.0 and 5.5 ms, 4 Gbases 35 and 22.2
//   bytes four at a time, 14             5.4 to 8.5 and 5.55     22 to 29 and 22.4
//   byte by byte, 16                     6.3 to 8.8 and 5.4      23 to 30 and 22.0
//   byte by byte, 14                     5.3 to 5.6 and 5.75     21.9 to 22.6 and 23.5
//   bytes four at a time, 12             5.5 and 6.0             22.3 and 24.6
// So bytes are taken one by one, and 16 wavefronts until a pass over regions used
// before shows too low a rate, then 14 for as long as the regions stay.
constexpr uint32_t STAGE_W16_LDS = 9 * 1280 - 2064;
static_assert(160 * 1024 / (STAGE_W16_LDS + 2064) == 14, "workgroups per CU");

// LDS layout of one tile (host and device agree through this struct).
struct TileGeom {
    uint32_t NW, NB;
    uint32_t off_px, off_pn, off_wv, off_wp, off_pk, off_inv, off_fwd, off_seg, off_ok, off_last, off_g;
    uint32_t bytes;
};

// Per window the low 32 bits of its minimum (all a record needs: unique bit,
// bucket, second bucket and unit bits) and the minimizer's offset in the
// window as a byte, per m-mer its strand as a bit; each lane's 16 entries are
// padded by one word so that lanes' accesses hit distinct LDS banks.  Other
// than tile_w16 also passes prefix minima through LDS (64-bit values, 4-bit
// positions), before the window minima are written over them.
__host__ __device__ inline TileGeom tile_geom(uint32_t T, uint32_t w, uint32_t k, uint32_t m) {
    TileGeom g;
    g.NW = T + tile_halo(w) + 1;
    // bases relative to borg: d0 in [1,16]; the furthest read is the word
    // after the one holding relative base d0 + max(TILE_MMERS+m-2, NW+k-2)
    uint32_t need = 48 + (TILE_MMERS + m > g.NW + k ? TILE_MMERS + m : g.NW + k);
    g.NB = (need + 31) / 32 * 32;
    uint32_t o = 0;
    g.off_g = o; o += GTAB_WORDS * 8;
    g.off_px = o;
    g.off_wv = o;
    g.off_wp = (o + 64 * 17 * 4 + 7) / 8 * 8;
    const bool lds_prefixes = !tile_w16(w, k);
    const uint32_t minima = g.off_wp + 64 * 20 + 4, prefixes = o + (lds_prefixes ? 64 * 17 * 8 : 0);
    o = ((minima > prefixes ? minima : prefixes) + 7) / 8 * 8;
    g.off_pn = o; o += lds_prefixes ? 64 * 8 : 0;
    g.off_pk = o; o += g.NB / 16 * 4;
    g.off_inv = o; o += (g.NB / 32 + 4) * 4;
    o = (o + 7) / 8 * 8;
    g.off_seg = o; o += (g.NW / 64 + 2) * 8;
    g.off_ok = o; o += (g.NW / 64 + 2) * 8;
    g.off_last = o; o += (g.NW / 64 + 2) * 8;
    g.off_fwd = o; o += 66 * 2;
    g.bytes = (o + 15) / 16 * 16;
    return g;
}

GG_DEV bool is_acgt(uint8_t c) {
    uint8_t u = c & 0xDF;
    return u == 'A' || u == 'C' || u == 'G' || u == 'T';
}

// Four bytes at a time.  2-bit codes (bits 1..2 of each letter) as 8 bits.
GG_DEV uint32_t codes4(uint32_t w) {
    const uint32_t x = (w >> 1) & 0x03030303u, y = (x << 6) | (x << 12);
    return (y | (y << 12)) >> 24;
}
// Bit j set when byte j of z is not zero.
GG_DEV uint32_t nonzero4(uint32_t z) {
    uint32_t f = (((z & 0x7F7F7F7Fu) + 0x7F7F7F7Fu) | z) & 0x80808080u;
    f |= f << 7;
    f |= f << 14;
    return f >> 28;
}
// Bit j set when byte j is none of ACGTacgt: bits 1..2 of a byte name its
// letter, whose bits 0 and 4 are those of 'A' for A, C and G and the opposite
// for T; bits 3, 6 and 7 are those of 'A' for all, bit 5 is the case.
GG_DEV uint32_t not_acgt4(uint32_t w) {
    const uint32_t t = (w >> 2) & ~(w >> 1) & 0x01010101u;
    return nonzero4((w ^ 0x41414141u ^ (t | (t << 4))) & 0xD9D9D9D9u);
}

struct Tile {
    const BucketArgs* A;
    TileGeom G;
    int64_t t0, wlo, borg;
    uint32_t d0;  // wlo - borg
    uint32_t* pk;
    uint32_t* inv;
    uint32_t* seg;
    uint32_t* ok;
    uint32_t* last;
    uint64_t* gt;
    uint64_t* px;  // prefix minima, entry i of lane q at 17 q + i (not tile_w16)
    uint64_t* pn;  // their positions in the lane's 16 m-mers, 4 bits each
    uint32_t* wv32;
    uint8_t* wp8;
    uint16_t* fwd16;

    GG_DEV uint32_t code_rel(int64_t r) const { return (pk[r >> 4] >> ((r & 15) * 2)) & 3; }
    GG_DEV bool inv_rel(int64_t r) const { return (inv[r >> 5] >> (r & 31)) & 1; }
    GG_DEV bool bit(const uint32_t* a, uint32_t x) const { return (a[x >> 5] >> (x & 31)) & 1; }
    // window minimum (its low 32 bits), its m-mer position, and the strand
    // flag of m-mer p
    GG_DEV uint64_t wval(uint32_t x) const { return wv32[x + (x >> 4)]; }
    GG_DEV uint32_t wpos(uint32_t x) const { return x + wp8[x + 4 * (x >> 4)]; }
    GG_DEV bool fwd_at(uint32_t p) const { return ((fwd16[p >> 4] >> (p & 15)) & 1u) != 0; }
};

// Low 32 bits of hi:lo >> s, 0 <= s < 32 (one v_alignbit).
GG_DEV uint32_t shift_pair(uint32_t lo, uint32_t hi, uint32_t s) { return ((hi << 1) << (s ^ 31u)) | (lo >> s); }

// 16 codes of relative positions [r, r+16) packed (position r at bits 0..1), r
// >= -16; positions below 0 read as whatever lies in front of the codes.
GG_DEV uint32_t extract16(const Tile& t, int64_t r) {
    const int32_t i = (int32_t)r;
    const uint32_t* p = t.pk + (i >> 4);
    return shift_pair(p[0], p[1], (i & 15) * 2);
}

GG_DEV uint32_t rev_comp16(uint32_t x) {
    uint32_t y = __brev(x);
    y = ((y >> 1) & 0x55555555u) | ((y & 0x55555555u) << 1);
    return y ^ 0xAAAAAAAAu;
}

template <int B>
GG_DEV void tile_minima(Tile& t);
GG_DEV void tile_minima_w16(Tile& t);

// Phases 0-3: load, hash, window minima, per-window flags.  B == 0 selects
// the path of w == 16 (k = 31, m = 15 and other k - m == 16), whose neighbour
// values all come from the next lane; otherwise B is tile_block(w).
template <int B>
GG_DEV void tile_compute(Tile& t) {
    const BucketArgs& A = *t.A;
    const TileGeom& G = t.G;
    const uint32_t lane = threadIdx.x;

    for (uint32_t i = lane; i < GTAB_WORDS; i += 64) t.gt[i] = A.gtab[i];

    // ---- phase 0: bases -> 2-bit codes + invalid bits --------------------
    const uint32_t nchunk = G.NB / 16;
    for (uint32_t c = lane; c < nchunk; c += 64) {
        int64_t a = t.borg + (int64_t)c * 16;
        uint32_t packed = 0, invm = 0;
        if (a >= 0 && a + 16 <= (int64_t)A.n) {
            uint4 v = *reinterpret_cast<const uint4*>(A.seq + a);
            if constexpr (B == 0) {
                // byte by byte: its VALU work is what this variant can spare (see STAGE_W16_LDS)
                const uint32_t wds[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
                for (uint32_t idx = 0; idx < 16; idx++) {
                    const uint8_t ch = (uint8_t)(wds[idx >> 2] >> (8 * (idx & 3)));
                    packed |= (uint32_t)((ch >> 1) & 3) << (2 * idx);
                    invm |= (is_acgt(ch) ? 0u : 1u) << idx;
                }
            } else {
                packed = codes4(v.x) | codes4(v.y) << 8 | codes4(v.z) << 16 | codes4(v.w) << 24;
                invm = not_acgt4(v.x) | not_acgt4(v.y) << 4 | not_acgt4(v.z) << 8 | not_acgt4(v.w) << 12;
            }
        } else {
            for (uint32_t idx = 0; idx < 16; idx++) {
                int64_t p = a + idx;
                uint8_t ch = (p >= 0 && p < (int64_t)A.n) ? A.seq[p] : (uint8_t)'\n';
                packed |= (uint32_t)((ch >> 1) & 3) << (2 * idx);
                invm |= (is_acgt(ch) ? 0u : 1u) << idx;
            }
        }
        t.pk[c] = packed;
        reinterpret_cast<uint16_t*>(t.inv)[c] = (uint16_t)invm;
    }
    __syncthreads();

    if constexpr (B == 0)
        tile_minima_w16(t);
    else
        tile_minima<B>(t);
}

// 64 bits of a bit array starting at bit `r` (r >= 0).
GG_DEV uint64_t bits64(const uint32_t* a, int64_t r) {
    const uint32_t wi = (uint32_t)(r >> 5), sh = (uint32_t)(r & 31);
    const uint32_t w0 = a[wi], w1 = a[wi + 1], w2 = a[wi + 2];
    return (uint64_t)shift_pair(w0, w1, sh) | (uint64_t)shift_pair(w1, w2, sh) << 32;
}

// Phases 1-3 for w == 16 and k <= 47, one window block of 16 per lane (NWB <=
// 62 blocks of windows).  The lane owning window block q hashes
// m-mer blocks q and q+1 (rolling update, tables in LDS), takes suffix minima
// of block q and running prefix minima of block q+1; window q*16+i is the
// combination of the two (van Herk / Gil-Werman in registers).  The window
// flags of phase 3 are formed in the same pass from a 64-bit slice of the
// invalid-base bitmap and written as 16-bit pieces.
// Bound by the record part's atomics and 16-byte stores, one of each per record
// and all at random addresses: 20 G/s of each, as long as wavefronts do not come
// to them sooner (see STAGE_W16_LDS).  The hashes, minima and flags of tile_minima
// are 28 % fewer VALU instructions and would bring them sooner.
GG_DEV void tile_minima_w16(Tile& t) {
    const TileGeom& G = t.G;
    const uint32_t lane = threadIdx.x;
    const uint32_t m = t.A->m, k = t.A->k;
    const int64_t rb = (int64_t)t.d0;  // relative base of m-mer 0 (and of window 0)
    const ulonglong2* gt2 = reinterpret_cast<const ulonglong2*>(t.gt);
    const uint32_t q = lane, NWB = (G.NW + 15) / 16;
    const bool have = q < NWB;
    const uint32_t p0 = q * 16;
    uint32_t segm = 0, okm = 0, lastm = 0;
    bool need_prev = false;
    // the lane's first and last window minima (compared across lanes below)
    uint64_t first_v = 0, last_v = 0;
    uint32_t first_p = 0, last_p = 0;
    // every lane q <= NWB hashes m-mer block q once; lane q takes block q+1
    // from lane q+1 by a lane shift instead of hashing it again
    uint64_t sv[16], nv[16];
    uint32_t sp[16];
    uint32_t fbits = 0;
    if (q <= NWB) {
        uint64_t fw = 0, rc = 0;
        for (uint32_t j = 0; j + 1 < m; j++) {
            const ulonglong2 g = gt2[16 + t.code_rel(rb + p0 + j)];
            fw = rotl1_64(fw) ^ g.x;
            rc = rotr1_64(rc) ^ g.y;
        }
        const uint32_t inw = extract16(t, rb + p0 + m - 1);
        const uint32_t outw = extract16(t, rb + p0 - 1);
#pragma unroll
        for (int i = 0; i < 16; i++) {
            const uint32_t in = (inw >> (2 * i)) & 3u, out = (outw >> (2 * i)) & 3u;
            const ulonglong2 g = gt2[(i == 0 ? 16u : out * 4u) + in];
            fw = rotl1_64(fw) ^ g.x;
            rc = rotr1_64(rc) ^ g.y;
            const uint64_t mn = fw < rc ? fw : rc;
            sv[i] = (mn << 1) | (fw != rc ? 1ULL : 0ULL);
            sp[i] = p0 + i;
            fbits |= (fw < rc ? 1u : 0u) << i;
        }
        t.fwd16[q] = (uint16_t)fbits;  // strands of m-mers p0 .. p0 + 15
    } else {
#pragma unroll
        for (int i = 0; i < 16; i++) {
            sv[i] = 0;
            sp[i] = 0;
        }
    }
#pragma unroll
    for (int i = 0; i < 16; i++) nv[i] = lane_next64(sv[i]);  // every lane takes part
    if (have) {
#pragma unroll
        for (int i = 14; i >= 0; i--) mm_combine(sv[i], sp[i], sv[i + 1], sp[i + 1], sv[i], sp[i]);
        // invalid bits of relative bases rb + p0 - 1 .. rb + p0 + 62
        const uint64_t im = bits64(t.inv, rb + p0 - 1);
        const uint64_t kmask = (1ULL << (k - 1)) - 1;
        {
            const uint32_t p1 = p0 + 16;
            uint64_t pv = 0, prv = 0;
            uint32_t pp = 0, prp = 0;
            uint32_t offs[4] = {0u, 0u, 0u, 0u};  // minimizer offsets in the window, one byte each
            uint32_t* wv_q = t.wv32 + q * 17;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                const uint64_t v = nv[i];  // m-mer p1 + i
                uint64_t rv = sv[i];
                uint32_t rp = sp[i];
                if (i > 0) mm_combine(sv[i], sp[i], pv, pp, rv, rp);
                wv_q[i] = (uint32_t)rv;
                offs[i >> 2] |= (rp - (p0 + i)) << (8 * (i & 3));
                if (i == 0) {
                    first_v = rv;
                    first_p = rp;
                }
                if (i == 15) {
                    last_v = rv;
                    last_p = rp;
                }
                // flags of window x = p0 + i (bases rb + x .. rb + x + k - 2)
                const uint32_t x = p0 + i;
                if (x >= 1 && x < G.NW) {
                    const bool valid = ((im >> (i + 1)) & kmask) == 0;
                    const bool first = (im >> i) & 1;
                    const bool lst = (im >> (i + k)) & 1;
                    const bool okf = valid && !(first && lst);
                    if (okf) {
                        okm |= 1u << i;
                        if (lst) lastm |= 1u << i;
                        if (first) {
                            segm |= 1u << i;
                        } else if (i == 0) {
                            need_prev = true;
                        } else if (rv != prv || ((rv & 1) && rp != prp)) {
                            segm |= 1u << i;
                        }
                    }
                }
                prv = rv;
                prp = rp;
                if (i == 0) {
                    pv = v;
                    pp = p1;
                } else {
                    mm_combine(pv, pp, v, p1 + i, pv, pp);
                }
            }
            uint32_t* o4 = reinterpret_cast<uint32_t*>(t.wp8 + 20 * q);
#pragma unroll
            for (int j = 0; j < 4; j++) o4[j] = offs[j];
        }
    }
    // window p0 starts a group when its minimum differs from window p0 - 1,
    // the previous lane's last window (every lane takes part in the shift)
    const uint64_t prev_v = lane_prev64(last_v);
    const uint32_t prev_p = lane_prev32(last_p);
    if (need_prev && (prev_v != first_v || ((first_v & 1) && first_p != prev_p))) segm |= 1u;
    // bitmap words past the last block stay zero
    const uint32_t npieces = (G.NW / 64 + 2) * 4;
    for (uint32_t pc = q; pc < npieces; pc += 64) {
        const bool mine = pc == q && have;
        reinterpret_cast<uint16_t*>(t.seg)[pc] = mine ? (uint16_t)segm : 0;
        reinterpret_cast<uint16_t*>(t.ok)[pc] = mine ? (uint16_t)okm : 0;
        reinterpret_cast<uint16_t*>(t.last)[pc] = mine ? (uint16_t)lastm : 0;
    }
    __syncthreads();
}

// Canonical ntHashes of the lane's m-mers p0 .. p0 + 15 (rolling update, tables
// in LDS) as v = hash << 1 | !symmetric; returns their strand bits.
//   fw_i = rotl1(fw_{i-1}) ^ rotl(h(s_{i-1}), m) ^ h(s_{i+m-1})
//   rc_i = rotr1(rc_{i-1}) ^ rotr1(rc(s_{i-1})) ^ rotl(rc(s_{i+m-1}), m-1)
// with the "out" term dropped while the first m bases are fed.
// The hashes are kept as 32-bit halves: as 64-bit values the compiler rotates
// them with 64-bit shifts, four times an alignbit's cost each.
struct Halves {
    uint32_t lo, hi;
};
template <int N>
GG_DEV Halves rotl_xor(Halves x, uint64_t g) {
    return {shift_pair(x.hi, x.lo, 32 - N) ^ (uint32_t)g, shift_pair(x.lo, x.hi, 32 - N) ^ (uint32_t)(g >> 32)};
}
template <int N>
GG_DEV Halves rotr_xor(Halves x, uint64_t g) {
    return {shift_pair(x.lo, x.hi, N) ^ (uint32_t)g, shift_pair(x.hi, x.lo, N) ^ (uint32_t)(g >> 32)};
}
GG_DEV uint64_t whole(Halves x) { return (uint64_t)x.hi << 32 | x.lo; }

GG_DEV uint32_t hash_block16(const Tile& t, uint32_t p0, uint64_t* v) {
    const ulonglong2* gt2 = reinterpret_cast<const ulonglong2*>(t.gt);
    const int64_t rb = (int64_t)t.d0 + p0;
    const uint32_t m = t.A->m;
    Halves fw{0u, 0u}, rc{0u, 0u};
    // the first m - 1 bases two at a time, then the odd one
    for (uint32_t j0 = 0; j0 + 2 < m; j0 += 16) {
        uint32_t c = extract16(t, rb + j0);
        const uint32_t n = m - 1 - j0 < 16 ? (m - 1 - j0) / 2 : 8;
        for (uint32_t j = 0; j < n; j++) {
            const ulonglong2 g = gt2[20 + (c & 15u)];
            fw = rotl_xor<2>(fw, g.x);
            rc = rotr_xor<2>(rc, g.y);
            c >>= 4;
        }
    }
    if ((m & 1) == 0) {
        const ulonglong2 g = gt2[16 + t.code_rel(rb + m - 2)];
        fw = rotl_xor<1>(fw, g.x);
        rc = rotr_xor<1>(rc, g.y);
    }
    const uint32_t inw = extract16(t, rb + m - 1);
    const uint32_t outw = extract16(t, rb - 1);
    uint32_t fbits = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const uint32_t in = (inw >> (2 * i)) & 3u, out = (outw >> (2 * i)) & 3u;
        const ulonglong2 g = gt2[(i == 0 ? 16u : out * 4u) + in];
        fw = rotl_xor<1>(fw, g.x);
        rc = rotr_xor<1>(rc, g.y);
        const uint64_t f = whole(fw), r = whole(rc);
        const bool less = f < r;
        const Halves mn{less ? fw.lo : rc.lo, less ? fw.hi : rc.hi};
        v[i] = whole({(mn.lo << 1) | (uint32_t)(f != r), shift_pair(mn.lo, mn.hi, 31)});
        fbits |= (uint32_t)less << i;
    }
    return fbits;
}

// Flags of the lane's 16 windows x = p0 + i from the invalid-base bits alone,
// one bit per window: `ok` when the window (bases x .. x + k - 2) is all ACGT
// and not an isolated one of its run, `first` / `last` when the base before /
// behind it ends the run.  Bit j of im = base p0 - 1 + j is invalid; a window
// is bad when any of bits i + 1 .. i + k - 1 is set: an OR over k - 1 shifts,
// doubled, for the 16 windows at once.
GG_DEV void window_flags16(const Tile& t, uint32_t p0, uint32_t* ok, uint32_t* first, uint32_t* last) {
    const uint32_t k = t.A->k;
    const int64_t r = (int64_t)t.d0 + p0 - 1;
    const u128_t im = (u128_t)bits64(t.inv, r) | ((u128_t)bits64(t.inv, r + 64) << 64);
    u128_t bad = im >> 1;
    uint32_t len = 1;
    while (2 * len <= k - 1) {
        bad |= bad >> len;
        len *= 2;
    }
    if (len < k - 1) bad |= bad >> (k - 1 - len);
    const uint32_t f = (uint32_t)im & 0xFFFFu, l = (uint32_t)(im >> k) & 0xFFFFu;
    // windows 1 .. NW - 1 of the tile
    uint32_t in = p0 + 16 <= t.G.NW ? 0xFFFFu : p0 >= t.G.NW ? 0u : (1u << (t.G.NW - p0)) - 1u;
    if (p0 == 0) in &= ~1u;
    *ok = ~(uint32_t)bad & ~(f & l) & in;
    *first = f;
    *last = l;
}

// Whether a window's minimum differs from the one of the window before (its
// value, or its position when unique), as 0 or 1.
GG_DEV uint32_t window_differs(uint64_t v, uint32_t p, uint64_t before_v, uint32_t before_p) {
    return (uint32_t)(v != before_v) | ((uint32_t)v & (uint32_t)(p != before_p) & 1u);
}

// Bitmaps of the tile's windows from the lanes' 16-bit pieces; words past the
// last window are zero.
GG_DEV void write_bitmaps16(Tile& t, uint32_t segm, uint32_t okm, uint32_t lastm) {
    const uint32_t lane = threadIdx.x;
    const uint32_t npieces = (t.G.NW / 64 + 2) * 4;
    for (uint32_t pc = lane; pc < npieces; pc += 64) {
        const bool mine = pc == lane;
        reinterpret_cast<uint16_t*>(t.seg)[pc] = mine ? (uint16_t)segm : 0;
        reinterpret_cast<uint16_t*>(t.ok)[pc] = mine ? (uint16_t)okm : 0;
        reinterpret_cast<uint16_t*>(t.last)[pc] = mine ? (uint16_t)lastm : 0;
    }
}

// mm_combine by selects: its if / else becomes exec-mask branches, one to three
// per combination.
GG_DEV void mm_select(uint64_t av, uint32_t ap, uint64_t bv, uint32_t bp, uint64_t& rv, uint32_t& rp) {
    const bool b = bv < av;
    rv = (b ? bv : av) & (av == bv ? ~1ULL : ~0ULL);
    rp = b ? bp : ap;
}

// Phases 1-3 for any w >= B: lane q hashes m-mers 16q .. 16q + 15 and keeps
// the suffix minima of their blocks of B in registers; the blocks' prefix
// minima go to LDS.  Window x = 16q + i covers the suffix of its block from
// i, the blocks between (none for w < 2B except one where the window crosses
// two block ends, at most three for B = 16; a block's last prefix minimum is
// its minimum) and the prefix up to m-mer x + w - 1 (van Herk / Gil-Werman
// with a block that need not be w).  All index arithmetic on i is uniform, so
// each window costs one 64-bit LDS read and two or three combinations, on all
// 64 lanes; LDS arrays of every m-mer and one lane per block of w before.
// Bound by VALU issue (64-bit hashing and compares).  Staging pass of 0.9
// Gbases at w = 42: 22.1 -> 5.4 ms; of 0.24 Gbases at w = 33: 5.5 -> 1.4 ms;
// with selects for branches, two bases per step of the first hash and four
// input bytes at a time 5.4 -> 4.4 and 1.4 -> 1.2 ms.
template <int B>
GG_DEV void tile_minima(Tile& t) {
    const uint32_t q = threadIdx.x, p0 = 16 * q, w = t.A->w;
    uint64_t sv[16];
    uint32_t sp[16];
    t.fwd16[q] = (uint16_t)hash_block16(t, p0, sv);
    uint32_t okm, firstm, lastm;
    window_flags16(t, p0, &okm, &firstm, &lastm);
    lastm &= okm;
    {
        uint64_t pv = 0, nib = 0;
        uint32_t pp = 0;
#pragma unroll
        for (int i = 0; i < 16; i++) {
            sp[i] = i;
            if (i % B == 0) {
                pv = sv[i];
                pp = i;
            } else {
                mm_select(pv, pp, sv[i], i, pv, pp);
            }
            t.px[17 * q + i] = pv;
            nib |= (uint64_t)pp << (4 * i);
        }
        t.pn[q] = nib;
#pragma unroll
        for (int i = 14; i >= 0; i--)
            if (i % B != B - 1) mm_select(sv[i], sp[i], sv[i + 1], sp[i + 1], sv[i], sp[i]);
    }
    __syncthreads();
    // window minima: low words, offsets, and where a window's minimum differs
    // from the window before
    uint32_t rv32[16], offs[4] = {0u, 0u, 0u, 0u}, diffm = 0;
    uint64_t first_v = 0, last_v = 0, mv = 0;
    uint32_t first_p = 0, last_p = 0, mp = 0, n_mid = 0;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        uint64_t rv = sv[i];
        uint32_t rp = p0 + sp[i];
        const uint32_t e = i + w - 1;  // last m-mer of the window, relative to p0
        const uint32_t d = e / B - i / B;  // blocks from the window's first m-mer to its last
        if (B == 16) {
            // the blocks between only grow with i
            while (n_mid + 1 < d) {
                n_mid++;
                const uint32_t qb = q + n_mid < 64 ? q + n_mid : 63u;  // windows past the tile's are not used
                const uint64_t bv = t.px[17 * qb + 15];
                const uint32_t bp = 16 * qb + (uint32_t)(t.pn[qb] >> 60);
                if (n_mid == 1) {
                    mv = bv;
                    mp = bp;
                } else {
                    mm_select(mv, mp, bv, bp, mv, mp);
                }
            }
            if (n_mid) mm_select(rv, rp, mv, mp, rv, rp);
        } else if (d == 2) {
            const uint32_t z = (i / B + 1) * B + B - 1;
            const uint32_t qb = q + (z >> 4) < 64 ? q + (z >> 4) : 63u;
            mm_select(rv, rp, t.px[17 * qb + (z & 15)], 16 * qb + (uint32_t)((t.pn[qb] >> (4 * (z & 15))) & 15), rv, rp);
        }
        if (d) {
            const uint32_t qe = q + (e >> 4) < 64 ? q + (e >> 4) : 63u;
            mm_select(rv, rp, t.px[17 * qe + (e & 15)], 16 * qe + (uint32_t)((t.pn[qe] >> (4 * (e & 15))) & 15), rv, rp);
        }
        rv32[i] = (uint32_t)rv;
        offs[i >> 2] |= (rp - (p0 + i)) << (8 * (i & 3));
        if (i == 0) {
            first_v = rv;
            first_p = rp;
        } else {
            diffm |= window_differs(rv, rp, last_v, last_p) << i;
        }
        last_v = rv;
        last_p = rp;
    }
    // window p0 against the previous lane's last window
    diffm |= window_differs(first_v, first_p, lane_prev64(last_v), lane_prev32(last_p));
    const uint32_t segm = okm & (firstm | diffm);
    __syncthreads();  // the prefix minima were read: their LDS is reused
#pragma unroll
    for (int i = 0; i < 16; i++) t.wv32[17 * q + i] = rv32[i];
    uint32_t* o4 = reinterpret_cast<uint32_t*>(t.wp8 + 20 * q);
#pragma unroll
    for (int j = 0; j < 4; j++) o4[j] = offs[j];
    write_bitmaps16(t, segm, okm, lastm);
    __syncthreads();
}

// Sub-bucket of a window minimum: bucket = (h >> 1) mod 2^b for a unique
// minimizer, the duplicates bucket 2^b otherwise; second bucket = next sb bits
// (crates/assembler_minimizer_bucketing/src/lib.rs:218-255,
//  crates/hashes/src/cn_nthash.rs:135-142).
GG_DEV uint32_t sub_of(uint64_t v, uint32_t b, uint32_t sb) {
    uint32_t bucket = (v & 1) ? (uint32_t)((v >> 1) & ((1ULL << b) - 1)) : (1u << b);
    uint32_t second = (uint32_t)((v >> (b + 1)) & ((1ULL << sb) - 1));
    return (bucket << sb) | second;
}

// Physical unit: the sub-bucket refined by xb more minimizer bits (unique
// minimizers only; duplicates-bucket records keep one unit per sub-bucket).
GG_DEV uint32_t unit_of(uint64_t v, uint32_t b, uint32_t sb, uint32_t xb) {
    uint32_t extra = (v & 1) ? (uint32_t)((v >> (b + 1 + sb)) & ((1ULL << xb) - 1)) : 0u;
    return (sub_of(v, b, sb) << xb) | extra;
}

GG_DEV void tile_init(Tile& t, const BucketArgs* A, uint64_t tile, uint8_t* lds) {
    t.A = A;
    t.G = tile_geom(A->T, A->w, A->k, A->m);
    t.t0 = (int64_t)tile * A->T;
    t.wlo = t.t0 - tile_halo(A->w);
    int64_t bo = t.wlo - 1;
    t.borg = (bo >= 0) ? (bo / 16) * 16 : -(((-bo) + 15) / 16) * 16;
    t.d0 = (uint32_t)(t.wlo - t.borg);
    t.gt = reinterpret_cast<uint64_t*>(lds + t.G.off_g);
    t.px = reinterpret_cast<uint64_t*>(lds + t.G.off_px);
    t.pn = reinterpret_cast<uint64_t*>(lds + t.G.off_pn);
    t.pk = reinterpret_cast<uint32_t*>(lds + t.G.off_pk);
    t.inv = reinterpret_cast<uint32_t*>(lds + t.G.off_inv);
    t.wv32 = reinterpret_cast<uint32_t*>(lds + t.G.off_wv);
    t.wp8 = lds + t.G.off_wp;
    t.fwd16 = reinterpret_cast<uint16_t*>(lds + t.G.off_fwd);
    t.seg = reinterpret_cast<uint32_t*>(lds + t.G.off_seg);
    t.ok = reinterpret_cast<uint32_t*>(lds + t.G.off_ok);
    t.last = reinterpret_cast<uint32_t*>(lds + t.G.off_last);
}

// Group ends among the 16 windows of the lane's block that the tile owns
// (windows halo .. halo+T-1, absolute index below n).  Returns the mask and
// sets *x0 / *j0 (first window, relative and absolute) and *segm.
GG_DEV uint32_t lane_end_mask16(const Tile& t, uint32_t* x0, int64_t* j0, uint32_t* segm) {
    const uint32_t q = threadIdx.x, q0 = tile_halo(t.A->w) / 16;
    *x0 = q * 16;
    *j0 = t.wlo + (int64_t)q * 16;
    *segm = 0;
    if (q < q0 || q >= q0 + t.A->T / 16) return 0;
    const uint32_t sg = reinterpret_cast<const uint16_t*>(t.seg)[q];
    const uint32_t okm = reinterpret_cast<const uint16_t*>(t.ok)[q];
    const uint32_t lastm = reinterpret_cast<const uint16_t*>(t.last)[q];
    const uint32_t next = t.bit(t.seg, *x0 + 16) ? 1u : 0u;
    const int64_t left = (int64_t)t.A->n - *j0;
    const uint32_t vm = left >= 16 ? 0xFFFFu : (left <= 0 ? 0u : (1u << left) - 1u);
    *segm = sg & vm;
    return okm & (lastm | (sg >> 1) | (next << 15)) & vm;
}

// Code of the base at absolute position p (LDS when inside the tile, else HBM).
GG_DEV uint32_t code_abs(const Tile& t, int64_t p) {
    int64_t r = p - t.borg;
    if (r >= 0 && r < (int64_t)t.G.NB) return t.code_rel(r);
    return (t.A->seq[p] >> 1) & 3;
}
GG_DEV bool invalid_abs(const Tile& t, int64_t p) {
    if (p < 0 || p >= (int64_t)t.A->n) return true;
    int64_t r = p - t.borg;
    if (r >= 0 && r < (int64_t)t.G.NB) return t.inv_rel(r);
    return !is_acgt(t.A->seq[p]);
}

constexpr uint32_t NO_UNIT = 0xFFFFFFFFu;

// Color of the record starting at byte `start`: the last color range that
// starts at or before it.
GG_DEV uint32_t color_of(const BucketArgs& A, int64_t start) {
    uint32_t lo = 0, hi = A.n_colors;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (A.color_starts[mid] <= (uint64_t)start) lo = mid; else hi = mid;
    }
    return A.colors[lo];
}

// Packs the bases [start, end) (reverse complement when rc) into dst words,
// reading the tile's LDS codes where they cover the bases and the input
// otherwise.
GG_DEV void pack_bases(const Tile& t, int64_t start, int64_t end, bool rc, uint32_t* dst) {
    const uint32_t len = (uint32_t)(end - start);
    uint32_t acc = 0;
    for (uint32_t i = 0; i < len; i++) {
        const uint32_t cd = rc ? (code_abs(t, end - 1 - i) ^ 2u) : code_abs(t, start + i);
        acc |= cd << (2 * (i & 15));
        if ((i & 15) == 15 || i + 1 == len) {
            dst[i >> 4] = acc;
            acc = 0;
        }
    }
}

// Long record: bases to the pool, the slot holds length and pool offset.
// Returns false when the pool is full (the host retries with a larger one).
GG_DEV bool write_long(const BucketArgs& A, const Tile& t, uint32_t* out, int64_t start, int64_t end, bool rc,
                       uint32_t flags, uint32_t minpos) {
    const uint32_t len = (uint32_t)(end - start);
    const uint64_t words = (len + 15) / 16;
    const unsigned long long off = atomicAdd(A.pool_cursor, (unsigned long long)words);
    out[0] = (flags << 8) | (minpos << 10) | META_LONG | (rc ? META_RC : 0u);
    out[1] = len;
    out[2] = (uint32_t)off;
    out[3] = (uint32_t)(off >> 32);
    for (uint32_t q = 4; q < A.slot_words; q++) out[q] = 0;
    if (off + words > A.pool_cap) return false;
    pack_bases(t, start, end, rc, A.pool + off);
    return true;
}

// Counts a record in its unit and returns its rank there (records << 32 |
// k-mer occurrences in one 64-bit atomic); flags a unit whose k-mer count
// would carry into the record count.
GG_DEV void count_record(const BucketArgs& A, uint32_t unit, uint32_t nk, unsigned long long* old) {
    *old = atomicAdd(&A.unit_ck[unit], (1ULL << 32) | nk);
}
GG_DEV uint32_t rank_of(const BucketArgs& A, unsigned long long old, uint32_t nk) {
    if ((uint32_t)old + nk < (uint32_t)old) atomicOr(A.error_flag, 8u);
    return (uint32_t)(old >> 32);
}

// One record of a tile: everything the slot needs.
struct RecInfo {
    int64_t start, end;
    uint32_t unit, meta, nk;  // meta: flags << 8 | minpos << 10 | rc | cross marks (length added on write)
    bool rc, ok;
};

GG_DEV RecInfo rec_info(const Tile& t, uint32_t x) {
    const BucketArgs& A = *t.A;
    const uint32_t k = A.k, m = A.m;
    RecInfo r;
    r.ok = false;
    const int64_t bwin = t.wlo + (int64_t)x;
    // group start: latest group-start bit at or before x inside the tile
    int64_t a = -1;
    {
        // (the word of x or the one before it holds the start of most groups)
        int32_t wi = (int32_t)(x >> 5);
        const uint32_t m1 = t.seg[wi] & ((2u << (x & 31)) - 1u);
        uint32_t msk = m1;
        if (!m1 && wi > 0) msk = t.seg[--wi];
        while (msk == 0 && wi > 0) msk = t.seg[--wi];
        if (msk) a = t.wlo + (int64_t)wi * 32 + (31 - __clz(msk));
    }
    if (a < 0) return r;  // group starts before the halo: deferred
    const uint64_t v = t.wval(x);
    const bool unique = v & 1;
    const bool include_first = invalid_abs(t, a - 1);
    const bool include_last = t.bit(t.last, x);
    r.start = include_first ? a : a - 1;
    r.end = include_last ? bwin + k - 1 : bwin + k;
    const uint32_t prel = t.wpos(x);
    const int64_t mmabs = t.wlo + prel;
    r.rc = A.canonical && unique && !t.fwd_at(prel);
    uint32_t minpos = 0;
    if (unique) minpos = r.rc ? (uint32_t)(r.end - mmabs - m) : (uint32_t)(mmabs - r.start);
    const uint32_t flags = ((include_first ? 1u : 0u) << (r.rc ? 1 : 0)) | ((include_last ? 1u : 0u) << (r.rc ? 0 : 1));
    const uint32_t sub = sub_of(v, A.b, A.sb);
    r.unit = unit_of(v, A.b, A.sb, A.xb);
    // Boundary k-mers shared with a neighbouring group of the same
    // sub-bucket that was scattered to another unit: the merge must combine
    // the two halves (cross marks, in stored orientation).  A unique group
    // spans at most w windows, so window a-1 is inside the halo.
    uint32_t cross = 0;
    if (unique && A.xb) {
        if (!include_first) {
            const uint64_t vl = t.wval((uint32_t)(a - t.wlo - 1));
            if (sub_of(vl, A.b, A.sb) == sub && unit_of(vl, A.b, A.sb, A.xb) != r.unit) cross |= r.rc ? META_XEND : META_XBEGIN;
        }
        if (!include_last) {
            const uint64_t vr = t.wval(x + 1);
            if (sub_of(vr, A.b, A.sb) == sub && unit_of(vr, A.b, A.sb, A.xb) != r.unit) cross |= r.rc ? META_XBEGIN : META_XEND;
        }
    }
    r.meta = (flags << 8) | (minpos << 10) | (r.rc ? META_RC : 0u) | cross;
    r.nk = (uint32_t)(r.end - r.start) - k + 1;
    r.ok = true;
    return r;
}

// Writes the slot of record r to out (16-byte aligned, slot_words words).
// Returns false when a long record did not fit the pool.
GG_DEV bool write_record(const Tile& t, const RecInfo& r, uint32_t* out) {
    const BucketArgs& A = *t.A;
    const uint32_t SW = A.slot_words;
    const uint32_t inline_cap = (SW - 1) * 16;
    const uint32_t len = (uint32_t)(r.end - r.start);
    const int64_t rs = r.start - t.borg;
    if (len <= inline_cap && rs >= 0) {
        // 16-byte stores (slots are a multiple of 4 words)
        const uint32_t nw = (len + 15) / 16;
        uint4* o4 = reinterpret_cast<uint4*>(out);
        for (uint32_t g = 0; g < SW / 4; g++) {
            uint32_t w4[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; j++) {
                const uint32_t q = 4 * g + j;
                uint32_t wq = 0;
                if (q == 0) {
                    wq = len | r.meta;
                } else if (q - 1 < nw) {
                    const uint32_t qi = q - 1;
                    if (!r.rc) {
                        wq = extract16(t, rs + 16 * qi);
                    } else {
                        wq = rev_comp16(extract16(t, (r.end - t.borg) - 16 * (int64_t)qi - 16));
                    }
                    const uint32_t rem = len - 16 * qi;
                    if (rem < 16) wq &= (1u << (2 * rem)) - 1u;
                }
                w4[j] = wq;
            }
            o4[g] = make_uint4(w4[0], w4[1], w4[2], w4[3]);
        }
        return true;
    }
    if (len > inline_cap) return write_long(A, t, out, r.start, r.end, r.rc, (r.meta >> 8) & 3u, (r.meta >> 10) & 0xFFu);
    // bases start before the tile's loaded range
    out[0] = len | r.meta;
    for (uint32_t q = 1; q < SW; q++) out[q] = 0;
    pack_bases(t, r.start, r.end, r.rc, out + 1);
    return true;
}

// Slot words (up to 8) of an inline record whose bases are in the tile's
// LDS, built in registers; false when the record takes the generic path
// (write_record: long records, bases before the tile, slots above 8 words).
GG_DEV bool record_words(const Tile& t, const RecInfo& r, uint4* w4) {
    const BucketArgs& A = *t.A;
    const uint32_t SW = A.slot_words;
    const uint32_t len = (uint32_t)(r.end - r.start);
    const int64_t rs = r.start - t.borg;
    if (SW > 8 || len > (SW - 1) * 16 || rs < 0) return false;
    // Word q holds 16 bases from rs + 16 q, or the reverse complement of the 16
    // before the end less 16 q.  Words past the record's bases are zero: they
    // read codes in the tile or, up to 7 words behind them, the invalid bits.
    const int32_t first = (int32_t)(r.rc ? r.end - t.borg - 16 : rs), step = r.rc ? -16 : 16;
    uint32_t wv[8];
    wv[0] = len | r.meta;
#pragma unroll
    for (uint32_t q = 0; q < 7; q++) {
        wv[q + 1] = 0;
        if (q < 3 || SW == 8) {
            const int32_t p = first + step * (int32_t)q, rem = (int32_t)len - 16 * (int32_t)q;
            const uint32_t x = extract16(t, p > -16 ? p : -16), y = rev_comp16(x);
            const uint32_t keep = rem >= 16 ? ~0u : (1u << (2 * (rem > 0 ? rem : 0))) - 1u;
            wv[q + 1] = (r.rc ? y : x) & keep;
        }
    }
    w4[0] = make_uint4(wv[0], wv[1], wv[2], wv[3]);
    w4[1] = make_uint4(wv[4], wv[5], wv[6], wv[7]);
    return true;
}

// Where record `rank` of `unit` goes: its region slot, or the next spill
// entry (nullptr when the spill list is full: the host retries with the
// counted size).  *color_at receives the matching color entry.
GG_DEV uint32_t* record_dest(const BucketArgs& A, uint32_t unit, uint32_t rank, uint32_t** color_at) {
    const uint32_t SW = A.slot_words;
    if (rank < A.unit_cap) {
        const uint64_t slot = (uint64_t)unit * A.unit_cap + rank;
        *color_at = A.region_color ? A.region_color + slot : nullptr;
        return A.region + slot * SW;
    }
    const uint32_t stripe = blockIdx.x & (A.spill_stripes - 1);
    unsigned long long pos = atomicAdd(A.spill_cursor + stripe * SPILL_STRIDE, 1ULL);
    *color_at = nullptr;
    if (pos >= A.spill_cap) return nullptr;
    pos += stripe * A.spill_cap;
    A.spill_unit[pos] = unit;
    A.spill_rank[pos] = rank;
    if (A.spill_color) *color_at = A.spill_color + pos;
    return A.spill_slots + pos * SW;
}

// Records handled per lane and pass of the record loop; their unit atomics
// are all in flight while their slot words are built.
constexpr uint32_t STAGE_R = 2;

// Pass 1 (one wavefront per tile): window minima and group ends; every record
// whose group starts inside the tile or its halo is counted in its unit
// (which gives its rank there), built and staged at the tile's positions; the
// first record of a tile whose group starts further back is deferred to
// bucket_defer_kernel, which runs once the group-start bitmap is complete.
template <int B>
__global__ __launch_bounds__(64) void bucket_stage_kernel(BucketArgs A) {
    extern __shared__ __align__(16) uint8_t lds[];
    Tile t;
    tile_init(t, &A, A.tile0 + blockIdx.x, lds);
    tile_compute<B>(t);
    const uint32_t lane = threadIdx.x;
    const uint32_t SW = A.slot_words;
    __shared__ uint16_t ends[1024];
    __shared__ uint32_t n_ends;
    {
        uint32_t x0, segm;
        int64_t j0;
        uint32_t endm = lane_end_mask16(t, &x0, &j0, &segm);
        if (j0 >= t.t0 && j0 < t.t0 + A.T) reinterpret_cast<uint16_t*>(A.seg_bits)[j0 >> 4] = (uint16_t)segm;
        const uint32_t cnt = __popc(endm);
        uint32_t inc = cnt;
        for (uint32_t d = 1; d < 64; d <<= 1) {
            const uint32_t y = __shfl_up(inc, d);
            if (lane >= d) inc += y;
        }
        uint32_t o = inc - cnt;
        while (endm) {
            const uint32_t i = __ffs(endm) - 1;
            endm &= endm - 1;
            ends[o++] = (uint16_t)(x0 + i);
        }
        if (lane == 63) n_ends = inc;
        __syncthreads();
    }
    const uint32_t n_end = n_ends;
    for (uint32_t e0 = 0; e0 < n_end; e0 += 64 * STAGE_R) {
        RecInfo ri[STAGE_R];
        unsigned long long old[STAGE_R];
#pragma unroll
        for (uint32_t r = 0; r < STAGE_R; r++) {
            const uint32_t ei = e0 + 64 * r + lane;
            ri[r].ok = false;
            old[r] = 0;
            if (ei >= n_end) continue;
            const uint32_t x = ends[ei];
            ri[r] = rec_info(t, x);
            if (ri[r].ok) {
                count_record(A, ri[r].unit, ri[r].nk, &old[r]);
            } else {
                // group starts before the halo (non-unique minimizer): defer
                const uint32_t d = atomicAdd(A.defer_count, 1u);
                if (d < A.n_tiles) {
                    A.defer[3 * (uint64_t)d] = (uint64_t)(t.wlo + (int64_t)x);
                    A.defer[3 * (uint64_t)d + 1] = t.wval(x);
                    A.defer[3 * (uint64_t)d + 2] = t.bit(t.last, x) ? 1 : 0;
                } else {
                    atomicOr(A.error_flag, 4u);
                }
            }
        }
        uint4 wv[STAGE_R][2];
        bool in_regs[STAGE_R];
#pragma unroll
        for (uint32_t r = 0; r < STAGE_R; r++) in_regs[r] = ri[r].ok && record_words(t, ri[r], wv[r]);
        // every rank, then every store of a record that takes its region slot,
        // then whatever reads memory: one counter orders loads, atomics and
        // stores, so a wait between two stores waits for the first of them
        uint32_t rank[STAGE_R];
        bool done[STAGE_R];
#pragma unroll
        for (uint32_t r = 0; r < STAGE_R; r++) rank[r] = ri[r].ok ? rank_of(A, old[r], ri[r].nk) : 0u;
#pragma unroll
        for (uint32_t r = 0; r < STAGE_R; r++) {
            done[r] = in_regs[r] && rank[r] < A.unit_cap;
            if (!done[r]) continue;
            uint4* o4 = reinterpret_cast<uint4*>(A.region + ((uint64_t)ri[r].unit * A.unit_cap + rank[r]) * SW);
            o4[0] = wv[r][0];
            if (SW == 8) o4[1] = wv[r][1];
        }
        if (A.region_color) {
#pragma unroll
            for (uint32_t r = 0; r < STAGE_R; r++)
                if (done[r]) A.region_color[(uint64_t)ri[r].unit * A.unit_cap + rank[r]] = color_of(A, ri[r].start);
        }
        // spilled, long and other records
#pragma unroll
        for (uint32_t r = 0; r < STAGE_R; r++) {
            if (!ri[r].ok || done[r]) continue;
            uint32_t* color_at;
            uint32_t* out = record_dest(A, ri[r].unit, rank[r], &color_at);
            if (!out || !write_record(t, ri[r], out)) continue;  // spill list or pool full: retried
            if (color_at) *color_at = color_of(A, ri[r].start);
        }
    }
}

// Deferred records (group start before the tile's halo; only groups with a
// non-unique minimizer are that long): the group-start bitmap is complete
// now, so the start is the last group start at or before the end window.
// One thread per record; bases are read from the input; staged in the
// overflow region.
__global__ void bucket_defer_kernel(BucketArgs A) {
    const uint64_t i = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x;
    const uint64_t n_defer = *A.defer_count;
    if (i >= n_defer || i >= A.n_tiles) return;
    const int64_t bwin = (int64_t)A.defer[3 * i];
    const uint64_t v = A.defer[3 * i + 1];
    const bool include_last = A.defer[3 * i + 2] != 0;
    const uint32_t k = A.k, SW = A.slot_words, inline_cap = (SW - 1) * 16;
    int64_t gw = bwin >> 5;
    uint32_t gm = A.seg_bits[gw] & ((2u << (bwin & 31)) - 1u);
    while (gm == 0 && gw > 0) gm = A.seg_bits[--gw];
    if (!gm) {
        atomicOr(A.error_flag, 4u);
        return;
    }
    const int64_t a = gw * 32 + (31 - __clz(gm));
    const bool include_first = (a == 0) || !is_acgt(A.seq[a - 1]);
    const int64_t start = include_first ? a : a - 1;
    const int64_t end = include_last ? bwin + k - 1 : bwin + k;
    const uint32_t len = (uint32_t)(end - start);
    // a non-unique minimizer: forward orientation, no minimizer position
    const uint32_t flags = (include_first ? 1u : 0u) | ((include_last ? 1u : 0u) << 1);
    const uint32_t unit = unit_of(v, A.b, A.sb, A.xb);
    unsigned long long old;
    count_record(A, unit, len - k + 1, &old);
    uint32_t* color_at;
    uint32_t* out = record_dest(A, unit, rank_of(A, old, len - k + 1), &color_at);
    if (!out) return;  // spill list full: the host retries with the counted size
    Tile none;  // no LDS codes: every base comes from the input
    none.A = &A;
    none.borg = 0;
    none.G.NB = 0;
    bool ok = true;
    if (len > inline_cap) {
        ok = write_long(A, none, out, start, end, false, flags, 0);
    } else {
        out[0] = len | (flags << 8);
        for (uint32_t q = 1; q < SW; q++) out[q] = 0;
        pack_bases(none, start, end, false, out + 1);
    }
    if (ok && color_at) *color_at = color_of(A, start);
}

// Splits the packed per-unit counts into records and k-mer occurrences.
// Also sums the k-mer occurrences into total[0] and the records into
// total[1] (cleared by the reset kernel; blocks of 256 threads).
__global__ __launch_bounds__(256) void unit_split_kernel(const unsigned long long* ck, uint32_t* count, uint32_t* kmers,
                                                        uint32_t n, unsigned long long* total) {
    __shared__ unsigned long long part[4], rpart[4];
    unsigned long long sum = 0, rsum = 0;  // k-mer occurrences, records
    for (uint32_t u = blockIdx.x * blockDim.x + threadIdx.x; u < n; u += gridDim.x * blockDim.x) {
        const unsigned long long c = ck[u];
        count[u] = (uint32_t)(c >> 32);
        kmers[u] = (uint32_t)c;
        sum += (uint32_t)c;
        rsum += c >> 32;
    }
    for (uint32_t d = 32; d; d >>= 1) {
        sum += __shfl_down(sum, d);
        rsum += __shfl_down(rsum, d);
    }
    if ((threadIdx.x & 63) == 0) {
        part[threadIdx.x >> 6] = sum;
        rpart[threadIdx.x >> 6] = rsum;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        const unsigned long long t = part[0] + part[1] + part[2] + part[3];
        const unsigned long long r = rpart[0] + rpart[1] + rpart[2] + rpart[3];
        if (t) atomicAdd(total, t);
        if (r) atomicAdd(total + 1, r);
    }
}

// Records and bases per sub-bucket (sums over its 2^xb units).
__global__ void sub_totals_kernel(const uint32_t* unit_count, const uint32_t* unit_kmers, uint32_t n_sub, uint32_t xb,
                                  uint32_t k, uint64_t* records, uint64_t* bases) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n_sub) return;
    uint64_t r = 0, b = 0;
    for (uint32_t u = s << xb; u < (s + 1) << xb; u++) {
        r += unit_count[u];
        b += unit_kmers[u] + (uint64_t)unit_count[u] * (k - 1);
    }
    records[s] = r;
    bases[s] = b;
}

// Clears the cursors of pass 1 (a kernel, so the pass can be captured in a graph).
__global__ void bucket_reset_kernel(BucketArgs A) {
    if (threadIdx.x < SPILL_STRIPES) A.spill_cursor[threadIdx.x * SPILL_STRIDE] = 0;
    if (threadIdx.x == 0) {
        *A.pool_cursor = 0;
        A.kmer_total[0] = 0;
        A.kmer_total[1] = 0;
        *A.defer_count = 0;
        *A.error_flag = 0;
    }
}

// Pass 2a: identical records of a unit counted once, as the reference's
// compactor merges identical super-k-mers of a bucket
// (crates/minimizer_bucketing/src/compactor.rs:128-196: same bases, length
// and flags; multiplicities summed).  Identical super-k-mers share their
// minimizer, so all copies of a record live in one unit.  One workgroup per
// unit whose region holds 2..DEDUP_WIDE records: 64 threads for units of up to
// DEDUP_SMALL records, 256 above (two launches; the small one also passes the
// other units through).  The records are loaded into LDS with 16-byte loads,
// each is inserted into an LDS table keyed by its slot words and color, a
// record equal to an earlier inserted one adds to that one's multiplicity (up
// to MAX_MULT per stored record), and the stored records are written back, in
// region order, to the front of the region with multiplicity - 1 in their
// meta word.  Spilled records (rank >= unit_cap) are stored as they are.
constexpr uint32_t DEDUP_SMALL = 256;
constexpr uint32_t DEDUP_WIDE = 1024;

GG_DEV uint32_t slot_hash(const uint32_t* w, uint32_t sw, uint32_t color) {
    uint32_t h = 0x9E3779B9u ^ color;
    for (uint32_t i = 0; i < sw; i++) {
        h ^= w[i];
        h *= 0x85EBCA6Bu;
        h ^= h >> 13;
    }
    h *= 0xC2B2AE35u;
    return h ^ (h >> 16);
}

// Dynamic LDS of a dedup workgroup taking up to max_rec records: their slot
// words, then (colored builds) their colors.
__host__ __device__ inline uint32_t dedup_lds_bytes(uint32_t max_rec, uint32_t slot_words, bool colored) {
    return max_rec * slot_words * 4 + (colored ? max_rec * 4 : 0);
}

// NT threads per workgroup, units of LO < records <= HI (and, with PASS, the
// other units kept as they are, except those of (DEDUP_SMALL, DEDUP_WIDE]
// when the wide launch takes them).  At most 8 16-byte pieces per thread.
template <uint32_t NT, uint32_t LO, uint32_t HI, bool PASS>
GG_DEV void unit_dedup_body(const BucketArgs& A, uint32_t n_units, bool wide) {
    extern __shared__ __align__(16) uint8_t lds[];
    __shared__ uint32_t mult[HI];  // 0: a copy of another record
    __shared__ uint32_t table[2 * HI];  // record index + 1, 0 = free
    __shared__ uint32_t wave_n[NT / 64];
    __shared__ uint32_t folded_k;  // k-mer positions of the copies folded into earlier records
    constexpr uint32_t TABLE = 2 * HI;
    const uint32_t SW = A.slot_words, tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    uint32_t* rec = reinterpret_cast<uint32_t*>(lds);  // slot words
    uint32_t* col = rec + HI * SW;  // colored builds only
    // a region must also fit the registers that stage it: with 16-word slots
    // units of up to 128 records do
    auto mine = [&](uint32_t n) { return n > LO && n <= HI && n * (SW / 4) <= 8 * NT; };
    // a unit's region is loaded into registers while the previous unit is
    // processed
    uint4 p0 = {}, p1 = {}, p2 = {}, p3 = {}, p4 = {}, p5 = {}, p6 = {}, p7 = {};
#define GG_DEDUP_PREFETCH(UU, CNT)                                                                 \
    do {                                                                                           \
        const uint32_t n_ = (CNT) < A.unit_cap ? (CNT) : A.unit_cap;                               \
        if (mine(n_)) {                                                                            \
            const uint4* s_ = reinterpret_cast<const uint4*>(A.region + (uint64_t)(UU) * A.unit_cap * SW); \
            const uint32_t m_ = n_ * (SW / 4);                                                     \
            if (tid < m_) p0 = s_[tid];                                                            \
            if (tid + NT < m_) p1 = s_[tid + NT];                                                  \
            if (tid + 2 * NT < m_) p2 = s_[tid + 2 * NT];                                          \
            if (tid + 3 * NT < m_) p3 = s_[tid + 3 * NT];                                          \
            if (tid + 4 * NT < m_) p4 = s_[tid + 4 * NT];                                          \
            if (tid + 5 * NT < m_) p5 = s_[tid + 5 * NT];                                          \
            if (tid + 6 * NT < m_) p6 = s_[tid + 6 * NT];                                          \
            if (tid + 7 * NT < m_) p7 = s_[tid + 7 * NT];                                          \
        }                                                                                          \
    } while (0)
    uint32_t u = blockIdx.x;
    uint32_t cnt = u < n_units ? A.sub_count[u] : 0u;
    if (u < n_units) GG_DEDUP_PREFETCH(u, cnt);
    for (; u < n_units; u += gridDim.x) {
        const uint32_t n = cnt < A.unit_cap ? cnt : A.unit_cap;
        const uint32_t spilled = cnt - n;
        uint32_t* reg = A.region + (uint64_t)u * A.unit_cap * SW;
        uint32_t* regc = A.region_color ? A.region_color + (uint64_t)u * A.unit_cap : nullptr;
        const uint32_t un = u + gridDim.x;
        const uint32_t cnt_next = un < n_units ? A.sub_count[un] : 0u;
        if (!mine(n)) {
            // kept as it is (by the small launch for every unit the wide
            // launch does not take)
            if (PASS && tid == 0 && !(wide && n > DEDUP_SMALL && n <= DEDUP_WIDE)) {
                A.unit_dregion[u] = n;
                A.unit_dcount[u] = cnt;
                A.unit_skmers[u] = A.sub_kmers[u];
            }
            cnt = cnt_next;
            if (un < n_units) GG_DEDUP_PREFETCH(un, cnt);
            continue;
        }
        const uint32_t n4 = n * (SW / 4);
        uint4* r4 = reinterpret_cast<uint4*>(rec);
        if (tid < n4) r4[tid] = p0;
        if (tid + NT < n4) r4[tid + NT] = p1;
        if (tid + 2 * NT < n4) r4[tid + 2 * NT] = p2;
        if (tid + 3 * NT < n4) r4[tid + 3 * NT] = p3;
        if (tid + 4 * NT < n4) r4[tid + 4 * NT] = p4;
        if (tid + 5 * NT < n4) r4[tid + 5 * NT] = p5;
        if (tid + 6 * NT < n4) r4[tid + 6 * NT] = p6;
        if (tid + 7 * NT < n4) r4[tid + 7 * NT] = p7;
        for (uint32_t i = tid; i < n; i += NT) {
            if (regc) col[i] = regc[i];
            mult[i] = 1;
        }
        for (uint32_t i = tid; i < TABLE; i += NT) table[i] = 0;
        if (tid == 0) folded_k = 0;
        __syncthreads();
        // the next unit's records are in flight meanwhile
        cnt = cnt_next;
        if (un < n_units) GG_DEDUP_PREFETCH(un, cnt);
        uint32_t my_folded = 0;
        for (uint32_t i = tid; i < n; i += NT) {
            const uint32_t* w = rec + i * SW;
            if (w[0] & META_LONG) continue;  // pool records: bases elsewhere, kept as they are
            const uint32_t ci = regc ? col[i] : 0u;
            uint32_t slot = slot_hash(w, SW, ci) & (TABLE - 1);
            for (uint32_t probe = 0; probe < TABLE; probe++) {
                uint32_t cur = table[slot];
                if (cur == 0) {
                    cur = atomicCAS(&table[slot], 0u, i + 1);
                    if (cur == 0) break;  // first of its kind: stored
                }
                const uint32_t j = cur - 1;
                const uint32_t* o = rec + j * SW;
                bool eq = !regc || col[j] == ci;
                for (uint32_t q = 0; q < SW && eq; q++) eq = o[q] == w[q];
                if (eq) {
                    // a copy of record j: counted there while j has room
                    uint32_t m = mult[j];
                    while (m < MAX_MULT) {
                        const uint32_t seen = atomicCAS(&mult[j], m, m + 1);
                        if (seen == m) break;
                        m = seen;
                    }
                    if (m < MAX_MULT) {
                        mult[i] = 0;
                        my_folded += meta_len(w[0]) - A.k + 1;  // inserts this copy no longer makes
                    }
                    break;
                }
                slot = (slot + 1) & (TABLE - 1);
            }
        }
        // one LDS atomic per wavefront for the folded copies' k-mer positions
        for (uint32_t d = 32; d >= 1; d >>= 1) my_folded += __shfl_down(my_folded, d);
        if (lane == 0 && my_folded) atomicAdd(&folded_k, my_folded);
        __syncthreads();
        // stored records to the front of the region, in region order
        uint32_t placed = 0;
        for (uint32_t i0 = 0; i0 < n; i0 += NT) {
            const uint32_t i = i0 + tid;
            const uint32_t m = i < n ? mult[i] : 0u;
            const uint64_t bal = __ballot(m != 0);
            uint32_t before = 0, total = (uint32_t)__popcll(bal);
            if (NT > 64) {
                if (lane == 0) wave_n[wave] = total;
                __syncthreads();
                total = 0;
                for (uint32_t q = 0; q < NT / 64; q++) {
                    const uint32_t c = wave_n[q];
                    if (q < wave) before += c;
                    total += c;
                }
            }
            if (m) {
                const uint32_t dst = placed + before + (uint32_t)__popcll(bal & ((1ULL << lane) - 1));
                const uint32_t* w = rec + i * SW;
                uint32_t* d = reg + (uint64_t)dst * SW;
                d[0] = w[0] | ((m - 1) << META_MULT_SHIFT);
                for (uint32_t q = 1; q < SW; q++) d[q] = w[q];
                if (regc) regc[dst] = col[i];
            }
            placed += total;
            if (NT > 64) __syncthreads();  // wave_n is reused by the next step
        }
        if (tid == 0) {
            A.unit_dregion[u] = placed;
            A.unit_dcount[u] = placed + spilled;
            A.unit_skmers[u] = A.sub_kmers[u] - folded_k;
        }
        __syncthreads();  // LDS reused by the next unit
    }
#undef GG_DEDUP_PREFETCH
}

// wide: unit_dedup_wide_kernel runs too and takes the larger units
__global__ __launch_bounds__(64) void unit_dedup_kernel(BucketArgs A, uint32_t n_units, uint32_t wide) {
    unit_dedup_body<64, 1, DEDUP_SMALL, true>(A, n_units, wide != 0);
}

__global__ __launch_bounds__(256) void unit_dedup_wide_kernel(BucketArgs A, uint32_t n_units) {
    unit_dedup_body<256, DEDUP_SMALL, DEDUP_WIDE, false>(A, n_units, true);
}

// Pass 2b: each unit's stored region records (the region's first
// unit_dregion[u] slots) to their place in the dense unit-major arena; one
// wavefront per unit, 16-byte copies.
__global__ __launch_bounds__(256) void unit_compact_kernel(BucketArgs A, uint32_t n_units) {
    const uint32_t SW = A.slot_words;
    const uint32_t lane = threadIdx.x & 63;
    const uint32_t waves = gridDim.x * (blockDim.x >> 6);
    for (uint32_t u = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6); u < n_units; u += waves) {
        const uint32_t n = A.unit_dregion[u];
        const uint64_t o0 = A.sub_off[u];
        const uint4* src = reinterpret_cast<const uint4*>(A.region + (uint64_t)u * A.unit_cap * SW);
        uint4* dst = reinterpret_cast<uint4*>(A.slots + o0 * SW);
        const uint32_t n4 = n * (SW / 4);
        for (uint32_t i = lane; i < n4; i += 64) dst[i] = src[i];
        if (A.region_color)
            for (uint32_t i = lane; i < n; i += 64) A.slot_color[o0 + i] = A.region_color[(uint64_t)u * A.unit_cap + i];
    }
}

// Pass 2c: spilled records (rank >= unit_cap) after their unit's stored
// region records.  longest: the longest stripe's records.
__global__ void spill_place_kernel(BucketArgs A, uint64_t longest) {
    const uint32_t SW = A.slot_words;
    for (uint64_t e = blockIdx.x * (uint64_t)blockDim.x + threadIdx.x; e < longest * A.spill_stripes;
         e += (uint64_t)gridDim.x * blockDim.x) {
        const uint32_t stripe = (uint32_t)(e / longest);
        const uint64_t at = e - stripe * longest, i = stripe * A.spill_cap + at;
        if (at >= A.spill_cursor[stripe * SPILL_STRIDE]) continue;
        const uint32_t unit = A.spill_unit[i];
        const uint64_t slot = A.sub_off[unit] + A.unit_dregion[unit] + (A.spill_rank[i] - A.unit_cap);
        if (slot >= A.sub_off[unit + 1]) {
            atomicOr(A.error_flag, 1u);
            continue;
        }
        const uint4* src = reinterpret_cast<const uint4*>(A.spill_slots + i * SW);
        uint4* dst = reinterpret_cast<uint4*>(A.slots + slot * SW);
        for (uint32_t g = 0; g < SW / 4; g++) dst[g] = src[g];
        if (A.spill_color) A.slot_color[slot] = A.spill_color[i];
    }
}

// Device-wide exclusive scan of uint32 counts into uint64 offsets (n+1
// entries): per-chunk sums, one-block scan of the sums, per-chunk scan.
constexpr uint32_t SCAN_CHUNK = 4096;  // 1024 threads x 4 elements

GG_DEV uint64_t block_exclusive_scan(uint64_t v, uint64_t* tmp, uint64_t& total) {
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    uint64_t x = v;
    for (uint32_t d = 1; d < 64; d <<= 1) {
        uint64_t y = __shfl_up(x, d);
        if (lane >= d) x += y;
    }
    if (lane == 63) tmp[wave] = x;
    __syncthreads();
    if (wave == 0) {
        uint64_t s = lane < nw ? tmp[lane] : 0;
        for (uint32_t d = 1; d < 64; d <<= 1) {
            uint64_t y = __shfl_up(s, d);
            if (lane >= d) s += y;
        }
        if (lane < nw) tmp[lane] = s;
    }
    __syncthreads();
    uint64_t base = wave ? tmp[wave - 1] : 0;
    total = tmp[nw - 1];
    __syncthreads();
    return base + x - v;
}

__global__ __launch_bounds__(1024) void scan_reduce_kernel(const uint32_t* counts, uint64_t* partial, uint32_t n) {
    __shared__ uint64_t tmp[16];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_CHUNK;
    uint64_t s = 0;
    for (uint32_t q = 0; q < 4; q++) {
        uint64_t i = base + (uint64_t)q * 1024 + threadIdx.x;
        if (i < n) s += counts[i];
    }
    uint64_t total;
    block_exclusive_scan(s, tmp, total);
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

__global__ __launch_bounds__(1024) void scan_partials_kernel(uint64_t* partial, uint32_t nb) {
    __shared__ uint64_t tmp[16];
    uint64_t carry = 0;
    for (uint32_t c = 0; c < nb; c += 1024) {
        uint32_t i = c + threadIdx.x;
        uint64_t v = i < nb ? partial[i] : 0;
        uint64_t total;
        uint64_t ex = block_exclusive_scan(v, tmp, total);
        if (i < nb) partial[i] = carry + ex;
        carry += total;
    }
    if (threadIdx.x == 0) partial[nb] = carry;
}

__global__ __launch_bounds__(1024) void scan_apply_kernel(const uint32_t* counts, const uint64_t* partial,
                                                          uint64_t* off, uint32_t n, uint32_t nb) {
    __shared__ uint64_t tmp[16];
    const uint64_t base = (uint64_t)blockIdx.x * SCAN_CHUNK;
    // thread t owns elements base + 4t .. base + 4t + 3
    uint32_t c[4];
    uint64_t s = 0;
    for (uint32_t q = 0; q < 4; q++) {
        uint64_t i = base + 4ull * threadIdx.x + q;
        c[q] = i < n ? counts[i] : 0;
        s += c[q];
    }
    uint64_t total;
    uint64_t run = partial[blockIdx.x] + block_exclusive_scan(s, tmp, total);
    for (uint32_t q = 0; q < 4; q++) {
        uint64_t i = base + 4ull * threadIdx.x + q;
        if (i < n) off[i] = run;
        run += c[q];
    }
    if (blockIdx.x == nb - 1 && threadIdx.x == 0) off[n] = partial[nb];
}

}  // namespace gg
