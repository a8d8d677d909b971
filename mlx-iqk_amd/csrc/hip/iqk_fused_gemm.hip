// Fused dequant-in-MFMA grouped GEMM: the prefill contraction straight from
// the relayout streams (gfx950, fp16 MFMA, f32 accumulation).
//
// Reference: the prefill route dequantizes the whole stack to fp16
// (src/mlx_iqk/nn.py:155-169) and contracts it with mx.gather_mm over the
// sorted pairs (nn.py:221-238).  Here each workgroup decodes the weight rows
// it needs straight into MFMA operands, so a prefill reads the 2-bit streams
// (1122 B per 4096-wide IQ2_KS row) instead of writing and re-reading 8 KiB of
// fp16 per row.  IQ2_K's operands are the producer's fp16 weights bit for bit
// (the same four-entry tables).  IQ2_KS and IQ1_S_R4 scale each weight row by
// one fp16 d, so their operands are the exact products n = idx v (IQ1_S_R4:
// (2s+1)(g + shift)), fp16 without rounding, and d multiplies the row's f32
// sums once in the epilogue: a weight enters as d n instead of fp16(d n), and
// a one-hot activation row still yields fp16(d n), the producer's weight.
//
// Work list: as the grouped GEMM, with group g = expert g: the slots (pair
// rows) are sorted by expert, expert g owns [offs[g], offs[g+1]), and a block
// takes one M-tile of the list (64 slots) and one column block c (weight rows
// [256c, 256c + 256) of the requested row range).  XCD x (blocks b with
// b % 8 == x) takes a contiguous eighth of the M-tiles, each with all its
// column blocks one after another, so the column blocks of a tile share its
// activations in that XCD's L2 and an expert's M-tiles share its streams
// there (dealing M-tile 8i + x to XCD x instead fetched 1.32x the unique
// bytes from HBM, an expert's tiles landing on several XCDs).
//
// Tile (more than 16 slots; smaller ones take few_slots_tile): 512 threads,
// eight wavefronts.  Wavefront w owns weight rows
// 32w .. 32w+31 of the block (the 32 columns of v_mfma_f32_32x32x16_f16) for
// all 64 slots (two 32-row MFMA blocks): two 16-register accumulators, so a
// wavefront needs about 128 VGPRs and four fit per SIMD.
// Reduction steps of 128: lane (n, kg) = (l % 32, l / 32) decodes the 64
// weights of sub-blocks 2kg and 2kg+1 of the step (k = 128s + 64kg .. +64)
// of its row and feeds them to the step's eight MFMAs u as weights
// 8(u % 4) .. +7 of sub-block 2kg + u / 4, in the order (0,4,1,5,2,6,3,7) that
// the byte-split table lookup produces; the staged activations are permuted
// to match.  A lane thus builds its fp16 tables once per sub-block, and the
// MFMA's k index maps to the same weight for A and B.  The step's
// activations (64 slots x 128 fp16) are staged in LDS, double buffered, one
// barrier per step, and read one MFMA operand at a time; the code words of
// the next step are loaded while this one computes.  The block's scale planes
// (all 256 rows, whole reduction axis) are copied to LDS once, rows padded so
// the 32 rows a wavefront reads at once fall in distinct banks.
//
// IQ1_S_R4: the lane's two 32-weight blocks of a step bring their index bytes
// and qh words with the step's loads (no scale planes), and the grid sits in
// LDS as each entry's pool selectors (16 KiB); two grid entries expand like
// one 16-code word, with the block's pool of exact products (2s+1)(g +
// shift), the row's d applied to the sums as for IQ2_KS.

#include <algorithm>
#include <type_traits>

#include "iqk_device.h"
#include "iqk_host.h"
#include "iqk_pool.h"

#define IQK_GRID_STORAGE __constant__ static const __attribute__((aligned(16)))
#include "../iq1s_grid.h"

namespace iqk {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));

typedef float float16_t __attribute__((ext_vector_type(16)));

constexpr int kFusedWaves = 8;                   // wavefronts per block, 32 weight rows each
constexpr int kFusedThreads = 64 * kFusedWaves;
constexpr int kFusedBM = 64;                     // slots per block
constexpr int kFusedBN = 32 * kFusedWaves;       // weight rows per block
constexpr int kFusedKS = 128;                    // reduction elements per step
constexpr int kXStride = 2 * kFusedKS + 16;      // LDS bytes per staged activation row
constexpr int kXChunks = 2 * kFusedKS / 16;      // 16-byte chunks of a staged row per step
constexpr int kXRows = kFusedThreads / kXChunks; // rows one staging pass covers
constexpr int kXPer = kFusedBM / kXRows;         // staging passes a step
static_assert(kFusedBM % kXRows == 0 && kFusedThreads >= 256, "whole staging passes; the work-list scan needs 256 threads");
constexpr uint32_t kNoStore = 0x7fffffffu;         // a slot without an output row: above any (n_slots <= 2^30)
static_assert(kXRows == 32, "staging pass i is the 32-row MFMA slot block i");

struct FusedArgs {
    const uint16_t *x;
    const void *s0, *s1, *s2, *s3, *s4;
    const uint32_t *offs;  // [n_groups + 1]
    const uint32_t *xr, *yr;
    uint16_t *y;
    uint32_t N;         // output columns: weight rows row_start .. row_start + N of each expert
    uint32_t out_rows;  // rows per expert in the streams
    uint32_t row_start;
    uint32_t n_groups, n_slots, n_x_rows;
    // null, or the pairs' expert ids (64-bit: wide_ids), slot lists and offsets
    // then unused: each block finds its tile's pairs itself (count_pairs, list_pairs)
    const uint32_t *ids;
    uint32_t wide_ids, pairs_per_row;
    // the expert's full rows would take the wide tiles: no tile takes the
    // few-slot form, whose sums run in another order (see takes_wide_tiles)
    uint32_t wide_order;
};

// How a launch cuts a group's slots into tiles.
enum TileCut : int {
    kCut64 = 0,    // 64-slot tiles, the last one partial
    kCutWide = 1,  // 128-slot tiles, the last one if it holds more than 64
    kCutRest = 2,  // what kCutWide leaves: one tile of at most 64 slots, or none
};

constexpr uint32_t kWideBM = 128;  // slots of a wide tile

template <int CUT>
__device__ __forceinline__ uint32_t tiles_of(uint32_t slots) {
    const uint32_t rest = slots % kWideBM;
    if constexpr (CUT == kCut64) return (slots + kFusedBM - 1) / kFusedBM;
    if constexpr (CUT == kCutWide) return slots / kWideBM + (rest > uint32_t(kFusedBM) ? 1u : 0u);
    return rest != 0 && rest <= uint32_t(kFusedBM) ? 1u : 0u;
}

struct FusedScan {
    uint32_t wave[8], group, tile;
};

// The group of an XCD's nth tile, and the tile's number within it: XCD x takes
// tiles x ceil(T / 8) .. of the list's T, in group order.  False (uniformly)
// past its share.  Up to a group a thread, the sizes are loaded and scanned
// once, for T and the tile both.  size_of: a group's slots; share: ceil(T / 8).
template <int CUT, int THREADS, class SizeOf>
__device__ __forceinline__ bool claim_tile(SizeOf size_of, uint32_t n_groups, uint32_t xcd, uint32_t nth,
                                           FusedScan &ts, uint32_t &group, uint32_t &mtile, uint32_t &share) {
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const auto tiles_at = [&](uint32_t g) { return g < n_groups ? tiles_of<CUT>(size_of(g)) : 0u; };
    const bool once = n_groups <= uint32_t(THREADS);  // uniform
    uint32_t total = 0;
    if (!once) {
        uint32_t cnt = 0;
        for (uint32_t g = tid; g < n_groups; g += THREADS) cnt += tiles_at(g);
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) cnt += __shfl_xor(cnt, off, 64);
        if (lane == 0) ts.wave[wave] = cnt;
        __syncthreads();
#pragma unroll
        for (int w = 0; w < THREADS / 64; ++w) total += ts.wave[w];
        __syncthreads();  // the rounds below rewrite the totals
    }
    uint32_t carry = 0, tile = 0;
    for (uint32_t base = 0; base < n_groups; base += THREADS) {
        const uint32_t cnt = tiles_at(base + tid);
        uint32_t incl = cnt;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t up = __shfl_up(incl, off, 64);
            if (lane >= uint32_t(off)) incl += up;
        }
        if (lane == 63) ts.wave[wave] = incl;
        __syncthreads();
        uint32_t sum = 0, before = 0;
#pragma unroll
        for (uint32_t w = 0; w < uint32_t(THREADS / 64); ++w) {
            before += w < wave ? ts.wave[w] : 0u;
            sum += ts.wave[w];
        }
        if (once) total = sum;
        const uint32_t excl = carry + before + incl - cnt;
        share = (total + 7) / 8;
        tile = xcd * share + nth;
        if (nth >= share || tile >= total) return false;  // uniform
        if (tile - excl < cnt) {  // one thread's, of all rounds
            ts.group = base + tid;
            ts.tile = tile - excl;
        }
        carry += sum;
        __syncthreads();
        if (tile < carry) break;  // uniform: found
    }
    group = __builtin_amdgcn_readfirstlane(ts.group);  // uniform (read from LDS): the stream bases stay scalar
    mtile = __builtin_amdgcn_readfirstlane(ts.tile);
    return true;
}

// A block's scale planes in LDS.  IQ2_KS: scl u8 [K/64], sch u8 [K/256],
// sex u8 [K/256], dv f16 per row.  IQ2_K: scl u16 [K/64], sex u8 [K/128],
// dv f16 [K/256].  Row strides are padded to an odd number of dwords.
// IQ2_K at K = 4096 keeps its dv plane out of LDS (DV_IN_LDS false): with it
// the planes (52 KB for 256 rows) and the activations would fit one block a
// CU; without it (43 KB), two.  Its lanes load their super-block scales
// instead, one 32-bit word (two super-blocks) every four steps.
template <int MEMBER, int K>
struct FusedScales {
    static constexpr bool KS = MEMBER == IQ2_KS;
    static constexpr bool DV_IN_LDS = !(MEMBER == IQ2_K && K == 4096);
    static constexpr int SCL = KS ? K / 64 : K / 32;    // bytes per row
    static constexpr int HB = KS ? K / 256 : 0;
    static constexpr int EX = KS ? K / 256 : K / 128;
    static constexpr int DV = KS ? 2 : K / 128;
    static constexpr int pad(int b) { return b == 0 ? 0 : ((b + 3) / 4 % 2 ? (b + 3) / 4 * 4 : (b + 3) / 4 * 4 + 4); }
    static constexpr int SCL_S = pad(SCL), HB_S = pad(HB), EX_S = pad(EX), DV_S = pad(DV);
    uint8_t scl[kFusedBN * SCL_S];
    uint8_t hb[KS ? kFusedBN * HB_S : 4];
    uint8_t ex[kFusedBN * EX_S];
    uint8_t dv[DV_IN_LDS ? kFusedBN * DV_S : 4];
};

// Copy `rows` (1 .. kFusedBN) rows of a plane (BYTES a row, consecutive in
// global memory) into LDS rows of STRIDE bytes, in 32-bit units where the
// rows are whole dwords (every plane but IQ2_KS's per-row scale), else
// 16-bit units.  Straight-line: every thread issues all its loads, then all
// its stores, so the plane costs one memory latency; units past `rows`
// re-read the last unit and land in LDS rows nobody stores from.
template <int BYTES, int STRIDE>
__device__ __forceinline__ void copy_plane(const uint8_t *src, int rows, uint8_t *dst, int tid) {
    using Unit = std::conditional_t<BYTES % 4 == 0, uint32_t, uint16_t>;
    static_assert(BYTES % sizeof(Unit) == 0 && STRIDE % sizeof(Unit) == 0, "whole units a row");
    constexpr int UNITS_PER_ROW = BYTES / sizeof(Unit);
    constexpr int UNITS = kFusedBN * UNITS_PER_ROW;
    constexpr int PER = (UNITS + kFusedThreads - 1) / kFusedThreads;
    const int last = rows * UNITS_PER_ROW - 1;
    Unit v[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) v[i] = reinterpret_cast<const Unit *>(src)[min(tid + kFusedThreads * i, last)];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int u = tid + kFusedThreads * i;
        if (UNITS % kFusedThreads == 0 || u < UNITS) {
            const int r = u / UNITS_PER_ROW, c = u - r * UNITS_PER_ROW;
            *reinterpret_cast<Unit *>(dst + r * STRIDE + sizeof(Unit) * c) = v[i];
        }
    }
}

// IQ2_K's exact pool products n_c = v_c x m (m = nibble - 8 the scale index,
// v the alphabet), as fp16 pairs (word 0: n0 | n1 << 16, word 1: n2 | n3 <<
// 16), by (alphabet << 4 | nibble), each exact in fp16 (|n| <= 248), signed
// zeros included (a negative value times a zero index is -0).
struct Iq2kProducts {
    uint32_t w[2 * 32];
};

constexpr Iq2kProducts make_iq2k_products() {
    Iq2kProducts t{};
    constexpr int v[2][4] = {{-31, -13, 1, 17}, {-26, -8, 6, 22}};
    for (int alpha = 0; alpha < 2; ++alpha)
        for (int nib = 0; nib < 16; ++nib) {
            const int e = 16 * alpha + nib;
            const _Float16 m = _Float16(short(nib - 8));
            for (int c = 0; c < 4; ++c) {
                const _Float16 n = _Float16(short(v[alpha][c])) * m;
                t.w[2 * e + c / 2] |= uint32_t(__builtin_bit_cast(uint16_t, n)) << (16 * (c % 2));
            }
        }
    return t;
}

__constant__ const Iq2kProducts kIq2kProducts = make_iq2k_products();

// IQ1_S_R4's exact pool products n_c = (2s + 1) (g_c + shift), g = -1 .. 2,
// shift = 1/8 (negative when qh bit 15 is set), by qh bits 12-15 (s | sign
// << 3): at most 8 significant bits, so exact in fp16, and d x n rounded
// once is the producer's f32 chain d (2s+1) (g + shift) rounded once.
struct Iq1Products {
    uint32_t w[2 * 16];
};

constexpr Iq1Products make_iq1_products() {
    Iq1Products t{};
    for (int e = 0; e < 16; ++e) {
        const int s = e & 7, sign = e & 8 ? -1 : 1;
        for (int c = 0; c < 4; ++c) {
            const _Float16 n = _Float16(float((2 * s + 1) * (8 * (c - 1) + sign)) / 8.f);
            t.w[2 * e + c / 2] |= uint32_t(__builtin_bit_cast(uint16_t, n)) << (16 * (c % 2));
        }
    }
    return t;
}

// A four-entry fp16 table (n0 | n1 << 16, n2 | n3 << 16) as a v_perm pool:
// the low bytes of n0 .. n3, then their high bytes.
constexpr uint2_t split_pool(uint32_t n01, uint32_t n23) {
    return {(n01 & 0xffu) | ((n01 >> 8) & 0xff00u) | ((n23 & 0xffu) << 16) | ((n23 & 0xff0000u) << 8),
            ((n01 >> 8) & 0xffu) | ((n01 >> 16) & 0xff00u) | (((n23 >> 8) & 0xffu) << 16) | ((n23 >> 24) << 24)};
}

// IQ1_S_R4's products as pools.
struct Iq1Pools {
    uint2_t p[16];
};

constexpr Iq1Pools make_iq1_pools() {
    Iq1Pools t{};
    const Iq1Products q = make_iq1_products();
    for (int e = 0; e < 16; ++e) t.p[e] = split_pool(q.w[2 * e], q.w[2 * e + 1]);
    return t;
}

__constant__ const Iq1Pools kIq1Pools = make_iq1_pools();

// IQ2_KS's exact products n_c = v_c x idx as pools, by (alphabet << 5 |
// idx + 16): |n| <= 496, so each is exact in fp16 (a negative value times a
// zero index is -0, as in the producer's chain).
struct Iq2ksPools {
    uint2_t p[64];
};

constexpr Iq2ksPools make_iq2ks_pools() {
    Iq2ksPools t{};
    constexpr int v[2][4] = {{-31, -13, 1, 17}, {-26, -8, 6, 22}};
    for (int alpha = 0; alpha < 2; ++alpha)
        for (int i5 = 0; i5 < 32; ++i5) {
            const _Float16 m = _Float16(short(i5 - 16));
            uint32_t w[2] = {0u, 0u};
            for (int c = 0; c < 4; ++c) {
                const _Float16 n = _Float16(short(v[alpha][c])) * m;
                w[c / 2] |= uint32_t(__builtin_bit_cast(uint16_t, n)) << (16 * (c % 2));
            }
            t.p[32 * alpha + i5] = split_pool(w[0], w[1]);
        }
    return t;
}

__constant__ const Iq2ksPools kIq2ksPools = make_iq2ks_pools();

// The pool d x n_c from exact fp16 products n_c: one correctly rounded
// packed fp16 multiply a pair.  The producer's f32 chain forms the same exact
// product (at most 11 + 9 significant bits, so no f32 rounding) and rounds
// it to fp16 once, so the entries are equal bit for bit, signed zeros
// included.  The words pass as scalars: __builtin_bit_cast of a vector
// element (n.y of a uint2_t) reads the vector's first element in this
// compiler.
__device__ __forceinline__ Pool scale_products(uint32_t n01, uint32_t n23, _Float16 d) {
    const uint32_t p01 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, n01) * d);
    const uint32_t p23 = __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, n23) * d);
    return {perm(p23, p01, 0x06040200u), perm(p23, p01, 0x07050301u)};
}

// IQ2_K's pools of the four 16-weight words of one u16 scale word scw
// (nibble w: word w's index) and alphabet bits ab, under super-block scale dd.
__device__ __forceinline__ void iq2k_pools(uint32_t scw, uint32_t ab, _Float16 dd, const uint2_t *ptab, Pool *p) {
            // byte w: the table offset 8 (alpha_w << 4 | nibble_w) of word w; a
            // v_perm spreads the scale word's bytes to (b0, b0, b1, b1), shifts
            // put nibble w at bits 3-6 of byte w, and the multiply copies
            // alphabet bit w to bit 8w (no two copies meet, so no carries;
            // pinned, or it becomes a quarter-rate 32-bit multiply)
            const uint32_t scp = perm(scw, scw, 0x01010000u);
            uint32_t a8 = __umul24(ab, 0x204081u);
            asm volatile("" : "+v"(a8));
            const uint32_t kofs = ((scp << 3) & 0x00780078u) | ((scp >> 1) & 0x78007800u) | ((a8 & 0x01010101u) << 7);
            const uint8_t *tab = reinterpret_cast<const uint8_t *>(ptab);
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                const uint2_t n = *reinterpret_cast<const uint2_t *>(tab + ((kofs >> (8 * w)) & 0xffu));
                p[w] = scale_products(uint32_t(n.x), uint32_t(n.y), dd);
            }
}

// The v_perm tables of lane (row, kg) at step s, one per 16-weight word of
// its 64 weights: IQ2_KS sub-blocks 4s + 2kg + h (two words each), IQ2_K
// sub-blocks 8s + 4kg + w (one word each).  IQ2_KS's tables are its exact
// products idx v (the row scale d is applied to the sums), one LDS read of
// `ptab` by (alphabet, scale index): against forming d idx v in fp16 a step
// (two tables), the Zipf prefill's gate projection measured 381.1 -> 365.1
// us.  IQ2_K's are d n with n = v x m from `ptab`, its d being per
// super-block: the same fp16 products as the producer's f32 chain.  IQ2_K's
// super-block scale comes from the dv plane, or (no dv plane in LDS) from
// dvw, the lane's dv word of steps 4(s/4) .. +3 (scales of super-blocks
// 2(s/4) and 2(s/4)+1).
template <int MEMBER, int K>
__device__ __forceinline__ void fused_pools(const FusedScales<MEMBER, K> &sc, int row, int s, int kg, uint32_t dvw,
                                            const uint2_t *ptab, Pool *p) {
    using S = FusedScales<MEMBER, K>;
    if constexpr (MEMBER == IQ2_KS) {
        const uint32_t scl = sc.scl[row * S::SCL_S + 2 * s + kg];  // nibbles of sub-blocks 4s+2kg, +1
        const uint32_t hb = sc.hb[row * S::HB_S + (s >> 1)];
        const uint32_t ab = sc.ex[row * S::EX_S + (s >> 1)];
        const int bit = 4 * (s & 1) + 2 * kg;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            // alphabet << 5 | the 5-bit scale index (idx + 16)
            const uint32_t e = ((scl >> (4 * h)) & 15u) | (((hb >> (bit + h)) & 1u) << 4) | (((ab >> (bit + h)) & 1u) << 5);
            const uint2_t q = ptab[e];
            p[2 * h] = {q.x, q.y};
            p[2 * h + 1] = p[2 * h];
        }
    } else {
        const uint32_t scw = *reinterpret_cast<const uint16_t *>(sc.scl + row * S::SCL_S + 2 * (2 * s + kg));
        const uint32_t ab = (sc.ex[row * S::EX_S + s] >> (4 * kg)) & 15u;
        _Float16 dd;
        if constexpr (S::DV_IN_LDS)
            dd = half_of_bits(*reinterpret_cast<const uint16_t *>(sc.dv + row * S::DV_S + 2 * (s >> 1)));
        else
            dd = half_of_bits(dvw >> (16 * ((s >> 1) & 1)));
        iq2k_pools(scw, ab, dd, ptab, p);
    }
}

// IQ1_S_R4 at one step: blocks b = 0, 1 of the lane (index bytes q[b], qh
// word b of q.z).  Pools p[2b], p[2b+1] are block b's (the products
// (2s+1) (g + shift) from the LDS table `ptab`; the row scale d is applied
// to the sums: 394.9 -> 377.4 us on the Zipf prefill's gate projection
// against forming d (2s+1) (g + shift) a block), and sels[2b+t] holds the
// pool selectors of the block's 8-weight groups 2t and 2t+1, read whole from
// the block's LDS table of them (grid_selectors): no shifts and masks a step.
// Against 16-bit code words expanded by expand_word_paired (their selectors
// formed a step) the Zipf prefill's gate projection measured 390.4 -> 379.1
// us, bit-identical: 28 fewer VALU a step for four times the LDS bytes of
// the lookups.
__device__ __forceinline__ void fused_iq1(uint4_t q, const uint2_t *grid, const uint2_t *ptab, Pool *p,
                                          uint4_t *sels) {
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        const uint32_t qw = q[b], h = (q.z >> (16 * b)) & 0xffffu;
        // grid field 3 never occurs: four products, by qh bits 12-15
        const uint2_t n = ptab[(h >> 12) & 15u];
        p[2 * b] = {n.x, n.y};
        p[2 * b + 1] = p[2 * b];
        uint2_t c[4];
#pragma unroll
        for (int t = 0; t < 4; ++t) c[t] = grid[((qw >> (8 * t)) & 0xffu) | (((h >> (3 * t)) & 7u) << 8)];
        sels[2 * b] = uint4_t{c[0].x, c[0].y, c[1].x, c[1].y};
        sels[2 * b + 1] = uint4_t{c[2].x, c[2].y, c[3].x, c[3].y};
    }
}

struct FusedGrid {
    uint2_t sel[IQK_IQ1S_GRID_SIZE];  // grid_selectors of every grid entry, 16 KiB
};

// Pool selectors of one grid entry (positions i at bits 2i): (p0, p4, p1,
// p5) and (p2, p6, p3, p7), one position a byte.
__device__ __forceinline__ uint2_t grid_selectors(uint32_t x) {
    return {(x & 0x0303u) | ((x << 14) & 0x03030000u), ((x >> 4) & 0x0303u) | ((x << 10) & 0x03030000u)};
}

// The 16 weights of two grid entries from their selectors (sel.xy entry 0,
// sel.zw entry 1), in expand_word_paired's output order for the 16-code word
// of the two entries (dword 2j: positions j, j+4 of entry 0; dword 2j+1: of
// entry 1), so the MFMAs and the staged activations are the same as for a
// code word.
__device__ __forceinline__ void expand_sel_paired(uint4_t sel, Pool p, uint32_t *out) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const uint32_t e = sel[i];
        const uint32_t lo = perm(p.lo, p.lo, e), hi = perm(p.hi, p.hi, e);
        out[4 * (i & 1) + (i >> 1)] = perm(hi, lo, 0x05010400u);
        out[4 * (i & 1) + (i >> 1) + 2] = perm(hi, lo, 0x07030602u);
    }
}

// ---- tiles of few slots -----------------------------------------------------------

constexpr int kFewSlots = 16;  // slots up to which a tile takes the path below

__device__ __forceinline__ uint4_t buffer_u4(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}

// A buffer of `bytes` from p: loads past it return zeros.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buffer_of(const void *p, uint64_t bytes) {
    constexpr uint64_t kCap = 0xffffffffull;
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), 0, int(uint32_t(bytes < kCap ? bytes : kCap)),
                                             0x00020000);
}

// The stream planes from stacked row row0 on, as buffers that end with the
// stack: a lane addresses one by a 32-bit offset (no 64-bit address a lane
// and plane, which the path below has no registers for), and a row past the
// stack reads zeros.
template <int MEMBER, int K>
struct FewPlanes {
    static constexpr int COUNT = MEMBER == IQ1_S_R4 ? 2 : 4;
    static constexpr uint32_t ROW[4] = {MEMBER == IQ1_S_R4 ? K / 8 : K / 4,
                                        MEMBER == IQ1_S_R4 ? K / 16 : MEMBER == IQ2_KS ? K / 64 : K / 32,
                                        MEMBER == IQ2_KS ? K / 256 : K / 128, MEMBER == IQ2_KS ? K / 256 : K / 128};
    __amdgpu_buffer_rsrc_t p[COUNT];

    __device__ __forceinline__ FewPlanes(const FusedArgs &a, size_t row0) {
        const size_t rows = size_t(a.n_groups) * a.out_rows - row0;
        const void *s[4] = {a.s0, a.s1, a.s2, a.s3};
#pragma unroll
        for (int i = 0; i < COUNT; ++i) p[i] = buffer_of(static_cast<const uint8_t *>(s[i]) + row0 * ROW[i], rows * ROW[i]);
    }
};

// One lane's weights of one row over a chunk of 512 reduction elements, in
// the decode GEMV's layout: lane (n, g) = (l % 16, l / 16) of a 16-row block
// holds row n; in step s (256 elements) of the chunk it takes 64 weights, the
// IQ2 members' k = 256s + 64g .. +63, IQ1_S_R4's k = 128g + 64s .. +63, so the
// four lanes of a row read 64 contiguous code bytes an instruction.
template <int MEMBER, int K>
struct FewLane {
    uint4_t q[MEMBER == IQ1_S_R4 ? 1 : 2];  // code words (IQ1_S_R4: four blocks' index words)
    uint32_t sc[2];                         // IQ2_KS: scl word a step; IQ2_K: scale u16 of both steps (sc[0]); IQ1_S_R4: qh words
    uint32_t hb, ab;                        // IQ2_KS: sch, sex of both super-blocks; IQ2_K: dv pair, sex

    // chunk c of row `row` (of the planes' first), lane group g
    __device__ __forceinline__ void load(const FewPlanes<MEMBER, K> &pl, uint32_t row, int c, int g) {
        using P = FewPlanes<MEMBER, K>;
        if constexpr (MEMBER == IQ1_S_R4) {
            q[0] = buffer_u4(pl.p[0], row * P::ROW[0] + 16 * g, 64 * c);
            const uint2_t h = __builtin_amdgcn_raw_buffer_load_b64(pl.p[1], row * P::ROW[1] + 8 * g, 32 * c, 0);
            sc[0] = h.x;
            sc[1] = h.y;
        } else {
            q[0] = buffer_u4(pl.p[0], row * P::ROW[0] + 16 * g, 128 * c);
            q[1] = buffer_u4(pl.p[0], row * P::ROW[0] + 64 + 16 * g, 128 * c);
            if constexpr (MEMBER == IQ2_KS) {
                const uint2_t v = __builtin_amdgcn_raw_buffer_load_b64(pl.p[1], row * P::ROW[1], 8 * c, 0);
                sc[0] = v.x;
                sc[1] = v.y;
                hb = __builtin_amdgcn_raw_buffer_load_b16(pl.p[2], row * P::ROW[2], 2 * c, 0);
                ab = __builtin_amdgcn_raw_buffer_load_b16(pl.p[3], row * P::ROW[3], 2 * c, 0);
            } else {
                sc[0] = __builtin_amdgcn_raw_buffer_load_b16(pl.p[1], row * P::ROW[1] + 2 * g, 16 * c, 0);
                sc[1] = __builtin_amdgcn_raw_buffer_load_b16(pl.p[1], row * P::ROW[1] + 8 + 2 * g, 16 * c, 0);
                ab = __builtin_amdgcn_raw_buffer_load_b32(pl.p[2], row * P::ROW[2], 4 * c, 0);
                hb = __builtin_amdgcn_raw_buffer_load_b32(pl.p[3], row * P::ROW[3], 4 * c, 0);
            }
        }
    }

    // The v_perm tables of step s's four 16-weight words, and (IQ1_S_R4) the
    // words' pool selectors.
    __device__ __forceinline__ void tables(int s, int g, const uint2_t *ptab, const uint2_t *grid, Pool *p,
                                           uint4_t *sels) const {
        if constexpr (MEMBER == IQ1_S_R4) {
            fused_iq1(uint4_t{s ? q[0].z : q[0].x, s ? q[0].w : q[0].y, sc[s], 0u}, grid, ptab, p, sels);
        } else if constexpr (MEMBER == IQ2_KS) {
            const uint32_t scl = sc[s] >> (8 * g);  // nibbles of sub-blocks 2g, 2g+1
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int bit = 8 * s + 2 * g + h;
                const uint32_t e = ((scl >> (4 * h)) & 15u) | (((hb >> bit) & 1u) << 4) | (((ab >> bit) & 1u) << 5);
                const uint2_t v = ptab[e];
                p[2 * h] = {v.x, v.y};
                p[2 * h + 1] = p[2 * h];
            }
        } else {
            iq2k_pools(sc[s], (ab >> (16 * s + 4 * g)) & 15u, half_of_bits((hb >> (16 * s)) & 0xffffu), ptab, p);
        }
    }

    __device__ __forceinline__ uint32_t word(int s, int w) const { return q[MEMBER == IQ1_S_R4 ? 0 : s][w]; }
};

// LDS shape of a few-slot tile: ROWS staged rows, PC chunks of 512 elements a phase.
template <int ROWS, int PC>
struct FewShape {
    static constexpr int PHASE = 512 * PC;           // reduction elements staged at once
    static constexpr int STRIDE = 2 * PHASE + 16;    // LDS bytes per staged row
    static constexpr int BYTES = ROWS * STRIDE;
    static constexpr int UNITS = 2 * PHASE / 16;     // 16-byte units a row
};

// A tile of at most ROWS (8 or 16) slots against the block's 256 weight rows,
// on v_mfma_f32_16x16x32_f16.  Most experts of a batch or a short prompt have
// such tiles only, and the work is then one expansion of every routed weight
// beside one read of its streams.  The 32-slot MFMAs of the larger tiles ran
// half empty or worse there, and a barrier every 128 elements held all eight
// wavefronts to the slowest one's loads.  Here a wavefront (32 rows, two
// 16-row blocks sharing every A read) keeps a chunk of 512 elements in flight
// while it expands another, and the activations are staged by phases of PC
// chunks, as many as 64 KB hold (IQ1_S_R4, beside its grid: 32 KB): between
// two phases the wavefronts run free of one another.
//
// What bounds it: VALU issue more than anything else, 61 to 65% of a SIMD's
// time (MFMA 15 to 19).  Taking the loads out leaves 88% of the time, the MFMAs
// 86%, and 16-row wavefronts at six or eight a SIMD measured the same, as did
// loads of whole rows turned through LDS.  The line at 16 slots:
// two 16-slot blocks an operand measured 5% slower than one 32-slot MFMA
// (1024 tokens, uniform: 24 slots an expert).  Measured (the kernel alone, 256
// experts, top-6, uniform routing, IQ2_KS gate): 24 tokens 102 -> 84 us, 64
// 176 -> 144, 128 209 -> 171, 512 227 -> 207; Zipf(1.1) routing: IQ2_KS gate
// 64 tokens 112 -> 94, 512 243 -> 227, IQ1_S_R4 gate 143 -> 123 and 235 -> 205
// (128 and 512), IQ2_K down 166 -> 157 and 271 -> 254; 2048 tokens 386 -> 369,
// 377 -> 356, 430 -> 418.
template <int MEMBER, int K, int ROWS, int PC, class RowsOf>
__device__ __forceinline__ void few_slots_tile(const FusedArgs &a, RowsOf rows_of, uint8_t *xs, uint32_t *slot_dst,
                                               uint32_t *slot_x, const uint2_t *ptab, const uint2_t *grid, uint32_t m0, uint32_t gend,
                                               uint32_t n0, int rows_here, size_t row0, int tid) {
    constexpr bool IQ1 = MEMBER == IQ1_S_R4;
    using F = FewShape<ROWS, PC>;
    constexpr int CHUNKS = K / 512;
    static_assert(CHUNKS % 2 == 0 && CHUNKS % PC == 0, "chunks go in pairs, whole phases");
    const int wave = tid >> 6, l = tid & 63, n = l & 15, g = l >> 4;
    // rows 32 wave + 16 r + n; one past the range reads what follows it (zeros
    // past the stack) and is not stored
    using Lane = FewLane<MEMBER, K>;
    const FewPlanes<MEMBER, K> planes(a, row0);
    const uint32_t wrow = uint32_t(32 * wave + n);
    Lane cur[2], nxt[2];
#pragma unroll
    for (int r = 0; r < 2; ++r) cur[r].load(planes, wrow + 16 * r, 0, g);
    // each slot's activation row (bytes into x; past x's buffer, so zeros, if
    // it has none) and output row
    const uint32_t xbytes = a.n_x_rows * uint32_t(2 * K);  // below 4 GiB (the entry point)
    const __amdgpu_buffer_rsrc_t xbuf = buffer_of(a.x, xbytes);
    if (tid < kFewSlots) {
        const uint32_t xp = m0 + uint32_t(tid);
        uint32_t off = xbytes, dst = kNoStore;
        if (xp < gend) {
            uint32_t row, yrow;
            rows_of(xp, row, yrow);
            if (row < a.n_x_rows) off = row * uint32_t(2 * K);
            if (yrow < a.n_slots) dst = yrow | (row < a.n_x_rows ? 0x80000000u : 0u);  // else NaN
        }
        slot_dst[tid] = dst;
        slot_x[tid] = off;
    }
    const int live = int(min(gend - m0, uint32_t(ROWS)));
    // phase ph: units (16 bytes, in the paired order of expand_word_paired) of
    // the live rows, four loads in flight a thread.  IQ1_S_R4's chunks are
    // stored as the lanes take them: [step][lane group][64 elements].
    const auto stage = [&](int ph) {
        const int units = live * F::UNITS;
        for (int u0 = 0; u0 < units; u0 += 4 * kFusedThreads) {
            uint4_t v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int u = u0 + kFusedThreads * i + tid, row = u / F::UNITS, c = u % F::UNITS;
                if (row < live) v[i] = buffer_u4(xbuf, slot_x[row] + 16 * c, 2 * F::PHASE * ph);
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int u = u0 + kFusedThreads * i + tid, row = u / F::UNITS;
                int c = u % F::UNITS;
                if constexpr (IQ1) c = (c & ~63) | ((c & 8) << 2) | ((c & 48) >> 1) | (c & 7);
                if (row < live)
                    *reinterpret_cast<uint4_t *>(xs + row * F::STRIDE + 16 * c) =
                        uint4_t{perm(v[i].z, v[i].x, 0x05040100u), perm(v[i].z, v[i].x, 0x07060302u),
                                perm(v[i].w, v[i].y, 0x05040100u), perm(v[i].w, v[i].y, 0x07060302u)};
            }
        }
    };
    __syncthreads();  // the slots' rows, the tables
    stage(0);
    __syncthreads();

    float4_t acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    // a lane whose slot is past the tile's last reads one of its live rows:
    // its products reach only its own output row, never stored
    const uint8_t *abase = xs + min(n, max(live - 1, 0)) * F::STRIDE + 128 * g;
    const auto chunk = [&](int c, const Lane (&now)[2], Lane (&then)[2]) {
        if (c > 0 && c % PC == 0) {
            __syncthreads();  // every wavefront is done with the last phase
            stage(c / PC);
            __syncthreads();
        }
        if (c + 1 < CHUNKS) {
#pragma unroll
            for (int r = 0; r < 2; ++r) then[r].load(planes, wrow + 16 * r, c + 1, g);
        }
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            Pool p[2][4];
            uint4_t sels[2][IQ1 ? 4 : 1];
#pragma unroll
            for (int r = 0; r < 2; ++r) now[r].tables(s, g, ptab, grid, p[r], sels[r]);
            const int aoff = 1024 * (c % PC) + 512 * s;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                half8_t af[2];
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    af[h] = __builtin_bit_cast(half8_t, *reinterpret_cast<const uint4_t *>(abase + aoff + 32 * w + 16 * h));
#pragma unroll
                for (int r = 0; r < 2; ++r) {
                    uint32_t bw[8];
                    if constexpr (IQ1)
                        expand_sel_paired(sels[r][w], p[r][w], bw);
                    else
                        expand_word_paired(now[r].word(s, w), p[r][w], bw);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const half8_t bf =
                            __builtin_bit_cast(half8_t, uint4_t{bw[h], bw[2 + h], bw[4 + h], bw[6 + h]});
                        acc[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(af[h], bf, acc[r], 0, 0, 0);
                    }
                }
            }
        }
    };
#pragma unroll 1
    for (int c = 0; c < CHUNKS; c += 2) {
        chunk(c, cur, nxt);
        chunk(c + 1, nxt, cur);
    }

    // D (16x16): lane (n, g), register i holds slot 4g + i of weight row n
#pragma unroll
    for (int r = 0; r < 2; ++r) {
        const int lrow = 32 * wave + 16 * r + n;
        if (lrow >= rows_here) continue;
        float d = 1.f;  // the row scale of the sums; IQ2_K's scales are in its pools
        if constexpr (MEMBER == IQ2_KS) d = float(half_of_bits(static_cast<const uint16_t *>(a.s4)[row0 + lrow]));
        if constexpr (IQ1) d = float(half_of_bits(static_cast<const uint16_t *>(a.s2)[row0 + lrow]));
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t dst = slot_dst[4 * g + i];
            if (dst != kNoStore)
                a.y[size_t(dst & 0x7fffffffu) * a.N + n0 + lrow] =
                    (dst >> 31) ? uint16_t(float_to_half_bits(MEMBER == IQ2_K ? acc[r][i] : acc[r][i] * d)) : kHalfNaN;
        }
    }
}

// ---- a block's own routing --------------------------------------------------------

// Small calls (takes_own_routing) need no route launch: each block counts the
// pairs of every expert, finds its tile from the counts, and lists its tile's
// pairs.  That reads the ids (8 KB at most, from L2) in place of the offsets,
// and replaces two dependent loads of the slots' rows.
constexpr uint32_t kSelfPairs = 2 * kFusedThreads, kSelfExperts = kFusedThreads;

// Expert of each of the thread's pairs (0, with bit 31, for an id that names
// none; 0xffffffff past the last pair), and the experts' pair counts.
__device__ __forceinline__ void count_pairs(const FusedArgs &a, uint32_t *sizes, uint32_t (&key)[kSelfPairs / kFusedThreads],
                                            int tid) {
    sizes[tid] = 0;
    uint32_t id[kSelfPairs / kFusedThreads];
#pragma unroll
    for (uint32_t i = 0; i < kSelfPairs / kFusedThreads; ++i) {
        const uint32_t p = min(uint32_t(tid) + kFusedThreads * i, a.n_slots - 1u);
        id[i] = a.ids[p << a.wide_ids];
        if (a.wide_ids && a.ids[2 * p + 1]) id[i] = 0xffffffffu;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < kSelfPairs / kFusedThreads; ++i) {
        key[i] = id[i] < a.n_groups ? id[i] : 0x80000000u;
        if (uint32_t(tid) + kFusedThreads * i < a.n_slots)
            atomicAdd(&sizes[key[i] & 0x7fffffffu], 1u);
        else
            key[i] = 0xffffffffu;
    }
    __syncthreads();
}

// Pairs m0 .. m0 + kFusedBM - 1 of group g, in pair order, bit 31 where the id
// named no expert.  counts: a word a wavefront.
__device__ __forceinline__ void list_pairs(const FusedArgs &a, const uint32_t (&key)[kSelfPairs / kFusedThreads],
                                           uint32_t g, uint32_t m0, uint32_t *pairs, uint32_t *counts, int tid) {
    const int lane = tid & 63, wave = tid >> 6;
    uint32_t before = 0;  // of the earlier pieces
#pragma unroll
    for (uint32_t i = 0; i < kSelfPairs / kFusedThreads; ++i) {
        if (kFusedThreads * i >= a.n_slots) break;  // uniform
        const bool mine = key[i] != 0xffffffffu && (key[i] & 0x7fffffffu) == g;
        const uint64_t m = __ballot(mine);
        __syncthreads();  // the counts' last readers (the sizes', before the first)
        if (lane == 0) counts[wave] = uint32_t(__popcll(m));
        __syncthreads();
        uint32_t at = before;
#pragma unroll
        for (int w = 0; w < kFusedWaves; ++w) {
            if (w < wave) at += counts[w];
            before += counts[w];
        }
        at += __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), 0u)) - m0;
        if (mine && at < uint32_t(kFusedBM)) pairs[at] = (uint32_t(tid) + kFusedThreads * i) | (key[i] & 0x80000000u);
    }
    __syncthreads();
}

// SELF: each block finds its tile's pairs from a.ids (a kernel of its own, so
// the listed form's code is unchanged).
template <int MEMBER, int K, bool SELF>
__global__ __launch_bounds__(kFusedThreads) __attribute__((amdgpu_waves_per_eu(4)))
void fused_gemm_kernel(FusedArgs a) {
    constexpr bool IQ1 = MEMBER == IQ1_S_R4;
    using S = FusedScales<IQ1 ? IQ2_KS : MEMBER, K>;
    constexpr int STEPS = K / kFusedKS;
    // Steps a code-word group: IQ1_S_R4 4, the IQ2 members 1.  Two-step
    // groups for the IQ2 members measured within 1% (IQ2_K gate 404.4 ->
    // 402.6 us, IQ2_KS gate 381.9 -> 380.8 us with 32 bytes of spills at 128
    // VGPRs; IQ2_K at 2048 wide has no room for them): with one step a
    // group, a line of their code plane is loaded four times, not 8 or 16.
    constexpr int G = IQ1 ? 4 : 1;
    static_assert(STEPS % G == 0, "whole groups of steps");
    __shared__ FusedScan ts;
    // per slot of the tile: its output row, bit 31 set when its activations
    // are real (else its output row is NaN), or kNoStore
    __shared__ uint32_t slot_dst[kFusedBM];
    __shared__ uint32_t slot_x[kFewSlots];
    __shared__ uint32_t pairs[SELF ? kFusedBM : 1];
    __shared__ uint2_t ptab[MEMBER == IQ2_K ? 32 : IQ1 ? 16 : 64];  // pool products (IQ2_K) or pools
    // Phases of a few-slot tile: 64 KB of activations beside the tables leave
    // two blocks a CU; IQ1_S_R4's grid leaves room for 32 KB.
    constexpr int P8 = IQ1 ? 4 : 8, PC8 = P8 < K / 512 ? P8 : K / 512;
    using F8 = FewShape<8, PC8>;
    using F16 = FewShape<16, P8 / 2>;
    constexpr int GRID_BYTES = IQ1 ? int(sizeof(FusedGrid)) : 0;
    constexpr int XS_BYTES = 2 * kFusedBM * kXStride;
    constexpr int WIDE_BYTES = XS_BYTES + (IQ1 ? 0 : int(sizeof(S)));
    constexpr int FEW_BYTES = F16::BYTES;
    static_assert(F8::BYTES <= FEW_BYTES && XS_BYTES % 16 == 0, "LDS sized for every form");
    __shared__ __attribute__((aligned(16))) uint8_t smem[GRID_BYTES + (WIDE_BYTES > FEW_BYTES ? WIDE_BYTES : FEW_BYTES)];
    uint2_t *const grid = reinterpret_cast<uint2_t *>(smem);  // IQ1_S_R4
    uint8_t *const fxs = smem + GRID_BYTES;
    auto &xs = *reinterpret_cast<uint8_t (*)[2][kFusedBM * kXStride]>(fxs);
    S &sc = *reinterpret_cast<S *>(fxs + (IQ1 ? 0 : XS_BYTES));

    const int tid = threadIdx.x;
    const uint32_t ncb = (a.N + kFusedBN - 1) / kFusedBN;  // column blocks
    const uint32_t xcd = blockIdx.x & 7u, j = blockIdx.x >> 3, cblock = j % ncb;
    uint32_t *const sizes = reinterpret_cast<uint32_t *>(fxs);  // SELF: every group's, until the tile's pairs are listed
    uint32_t key[kSelfPairs / kFusedThreads];                   // SELF: of pairs tid + 512 i
    if constexpr (SELF) count_pairs(a, sizes, key, tid);
    const auto size_of = [&](uint32_t e) { return SELF ? sizes[e] : a.offs[e + 1] - a.offs[e]; };
    uint32_t g, mtile, share;
    if (!claim_tile<kCut64, kFusedThreads>(size_of, a.n_groups, xcd, j / ncb, ts, g, mtile, share)) return;  // surplus

    // Offsets and row indices are device data: a slot outside [0, n_slots)
    // is never stored, a row outside x is never read (its output row is NaN),
    // and a weight row past out_features is never stored.  Loads of such
    // rows read an in-bounds row instead, so the step has no branches but
    // (IQ1_S_R4) the one that skips staging activation rows past the tile's
    // end.
    // (SELF: slots count from the group's first)
    const uint32_t gend = SELF ? __builtin_amdgcn_readfirstlane(sizes[g]) : min(a.offs[g + 1], a.n_slots);
    const uint32_t m0 = (SELF ? 0u : a.offs[g]) + mtile * kFusedBM;
    if constexpr (SELF) list_pairs(a, key, g, m0, pairs, ts.wave, tid);
    // slot xp's activation row (none: past x) and output row
    const auto rows_of = [&](uint32_t xp, uint32_t &row, uint32_t &yrow) {
        if constexpr (SELF) {
            const uint32_t p = pairs[xp - m0];
            yrow = p & 0x7fffffffu;
            row = (p >> 31) ? a.n_x_rows : yrow / a.pairs_per_row;
        } else {
            row = a.xr[xp];
            yrow = a.yr ? a.yr[xp] : xp;
        }
    };
    const uint32_t n0 = cblock * kFusedBN;
    const int rows_here = int(min(uint32_t(kFusedBN), a.N - n0));
    const size_t row0 = size_t(g) * a.out_rows + a.row_start + n0;  // first stacked weight row of the block

    if constexpr (MEMBER == IQ2_K) {
        if (tid < 32) ptab[tid] = reinterpret_cast<const uint2_t *>(kIq2kProducts.w)[tid];
    } else if constexpr (IQ1) {
        if (tid < 16) ptab[tid] = kIq1Pools.p[tid];
    } else {
        if (tid < 64) ptab[tid] = kIq2ksPools.p[tid];
    }
    if constexpr (IQ1) {  // the grid as pool selectors
        static_assert(IQK_IQ1S_GRID_SIZE == 4 * kFusedThreads, "four grid entries a thread");
        const uint2_t cw = reinterpret_cast<const uint2_t *>(iqk_iq1s_grid_codes)[tid];
#pragma unroll
        for (int i = 0; i < 4; ++i)
            grid[4 * tid + i] = grid_selectors(((i < 2 ? cw.x : cw.y) >> (16 * (i & 1))) & 0xffffu);
    }
    // Few slots (uniform per block).  The empty asm keeps the forms' code
    // apart: merged ahead of the branches it costs each of them registers
    // (IQ1_S_R4, at 128 VGPRs, spills one or two even so).
    const uint32_t few = a.wide_order ? 0xffffffffu : gend - m0;
    if (few <= 8u) {
        asm volatile("" ::"n"(8));
        few_slots_tile<MEMBER, K, 8, PC8>(a, rows_of, fxs, slot_dst, slot_x, ptab, grid, m0, gend, n0, rows_here, row0, tid);
        return;
    }
    if (few <= uint32_t(kFewSlots)) {
        asm volatile("" ::"n"(16));
        few_slots_tile<MEMBER, K, 16, P8 / 2>(a, rows_of, fxs, slot_dst, slot_x, ptab, grid, m0, gend, n0, rows_here, row0, tid);
        return;
    }
    // scale planes of the block's rows
    if constexpr (!IQ1)
        copy_plane<S::SCL, S::SCL_S>(static_cast<const uint8_t *>(a.s1) + row0 * S::SCL, rows_here, sc.scl, tid);
    if constexpr (MEMBER == IQ2_KS) {
        copy_plane<S::HB, S::HB_S>(static_cast<const uint8_t *>(a.s2) + row0 * S::HB, rows_here, sc.hb, tid);
        copy_plane<S::EX, S::EX_S>(static_cast<const uint8_t *>(a.s3) + row0 * S::EX, rows_here, sc.ex, tid);
        copy_plane<S::DV, S::DV_S>(static_cast<const uint8_t *>(a.s4) + row0 * S::DV, rows_here, sc.dv, tid);
    } else if constexpr (MEMBER == IQ2_K) {
        copy_plane<S::EX, S::EX_S>(static_cast<const uint8_t *>(a.s2) + row0 * S::EX, rows_here, sc.ex, tid);
        if constexpr (S::DV_IN_LDS)
            copy_plane<S::DV, S::DV_S>(static_cast<const uint8_t *>(a.s3) + row0 * S::DV, rows_here, sc.dv, tid);
    }

    // activation staging: thread t moves 16-byte chunk t % kXChunks of slot
    // rows t / kXChunks + kXRows i a step, so the eight lanes of each LDS
    // store phase write 128 contiguous bytes (a thread's two chunks side by
    // side had every store phase hit each bank twice).  Byte offsets into x
    // are 32-bit (the entry point refuses an x of 4 GiB or more).
    // A row past the tile's last slot feeds only MFMA rows that are never
    // stored, so IQ1_S_R4 neither loads nor stages it per step (its LDS row
    // keeps the zeros written at the tile's start): a partial tile (most
    // tiles of a skewed routing) stages only its slots.  Measured on the 2048-token Zipf prefill:
    // IQ1_S_R4 -4%; the IQ2 members, whose step the branch splits for the
    // scheduler, +1 to +2%, so they stage every row.
    const int xrow_l = tid / kXChunks, xchunk = tid % kXChunks;
    const uint8_t *xbase = reinterpret_cast<const uint8_t *>(a.x);
    uint32_t xoff[kXPer];
    bool xlive[kXPer];
#pragma unroll
    for (int i = 0; i < kXPer; ++i) {
        const int row = xrow_l + kXRows * i;
        const uint32_t xp = m0 + uint32_t(row);
        uint32_t xrow = a.n_x_rows, yrow = kNoStore;
        if (xp < gend) rows_of(xp, xrow, yrow);
        const bool xv = xrow < a.n_x_rows;
        // a dead slot reads row 0 (the entry point refuses an empty x); its
        // products feed only its own output row, never stored as a value
        // chunks 8 .. 15 (lane group 1's half of a step) start 64G elements
        // after chunks 0 .. 7 in x, 64 in the staged row (see x_step)
        xoff[i] = (xv ? xrow : 0u) * uint32_t(2 * K) + uint32_t(16 * xchunk) + (xchunk >= 8 ? 128u * (G - 1) : 0u);
        xlive[i] = !IQ1 || xp < gend;
        if (xchunk == 0) {  // one thread a slot: the epilogue's destination, read once
            slot_dst[row] = yrow < a.n_slots ? yrow | (xv ? 0x80000000u : 0u) : kNoStore;
        }
    }
    // Staging pass i covers slot block i (rows 32i .. 32i+31): a tile of
    // MB slot blocks loads and stages passes 0 .. MB-1 only.
    // Steps go in groups of G (below): step Gp + j stages the 64 elements
    // from 128Gp + 64j (lane group 0's) and from 128Gp + 64G + 64j (lane
    // group 1's).
    const auto x_step = [&](int s) { return uint32_t(256 * G * (s / G) + 128 * (s % G)); };
    const auto load_x = [&](int s, uint4_t *v, auto passes) {
#pragma unroll
        for (int i = 0; i < decltype(passes)::value; ++i)
            if (xlive[i]) v[i] = load_u4(xbase + xoff[i] + x_step(s));
    };
    // Each 8-element chunk is stored in the order (0,4,1,5,2,6,3,7), the
    // order expand_word_paired gives the weights.  A row past the tile's last
    // slot is staged as zeros, so the MFMAs of those rows multiply zeros: the
    // kernel is bound by the clock its power allows, and zero operands draw
    // less (IQ2_KS gate 400.7 -> 392.5 us, IQ2_K gate 426.7 -> 417.0 us on
    // the 2048-token Zipf prefill; the rows were a dead slot's real data).
    // The IQ2 members stage every row, the dead ones through v_perm
    // selectors of 0x0c bytes (which give zero bytes: no instruction added);
    // IQ1_S_R4 zeroes its dead rows in both buffers once.
    uint32_t xsel_lo[kXPer], xsel_hi[kXPer];
#pragma unroll
    for (int i = 0; i < kXPer; ++i) {
        const bool dead = m0 + uint32_t(xrow_l + kXRows * i) >= gend;
        xsel_lo[i] = dead ? 0x0c0c0c0cu : 0x05040100u;
        xsel_hi[i] = dead ? 0x0c0c0c0cu : 0x07060302u;
        if (IQ1 && dead) {
#pragma unroll
            for (int b = 0; b < 2; ++b)
                *reinterpret_cast<uint4_t *>(xs[b] + (xrow_l + kXRows * i) * kXStride + 16 * xchunk) =
                    uint4_t{0u, 0u, 0u, 0u};
        }
    }
    const auto store_x = [&](int buf, const uint4_t *v, auto passes) {
        uint8_t *dst = xs[buf] + xrow_l * kXStride + 16 * xchunk;
#pragma unroll
        for (int i = 0; i < decltype(passes)::value; ++i)
            if (xlive[i])
                *reinterpret_cast<uint4_t *>(dst + kXRows * kXStride * i) =
                    uint4_t{perm(v[i].z, v[i].x, xsel_lo[i]), perm(v[i].z, v[i].x, xsel_hi[i]),
                            perm(v[i].w, v[i].y, xsel_lo[i]), perm(v[i].w, v[i].y, xsel_hi[i])};
    };

    // this lane's weight row and code words; a row past out_features reads
    // the block's first row.  The block's first row of each plane is a
    // uniform base, the lane's offsets from it are 32-bit (the entry point
    // refuses an expert plane of 4 GiB or more).  The steps go in groups of
    // G, lane group kg taking elements 128Gp + 64G kg .. +64G-1 of group p
    // (64j .. 64j+63 of those in its step j), so a lane loads its code bytes
    // once a group: IQ2 members 16G bytes (four words a step), IQ1_S_R4 (G =
    // 4) 32 bytes of index words and 16 of qh words.  A 128-byte line of a
    // code plane is then loaded 4/G times (IQ2; IQ1_S_R4 two and four times
    // against eight and sixteen with a load a step: 2.13x its unique bytes
    // fetched, 440.5 -> 411.9 us on the Zipf prefill gate).
    const int wave = tid >> 6, l = tid & 63, ln = l & 31, kg = l >> 5;
    const int lrow = 32 * wave + ln;
    const bool wv = lrow < rows_here;
    constexpr uint32_t QROW = IQ1 ? K / 8 : K / 4;  // code-plane bytes a row
    const uint8_t *qbase = static_cast<const uint8_t *>(a.s0) + row0 * QROW;
    const uint8_t *hbase = static_cast<const uint8_t *>(a.s1) + row0 * (K / 16);
    const uint32_t wl = wv ? uint32_t(lrow) : 0u;
    const uint32_t qoff = wl * QROW + uint32_t((IQ1 ? 8 : 16) * G * kg), hoff = wl * uint32_t(K / 16) + uint32_t(16 * kg);
    struct CodeGroup {
        uint4_t w[IQ1 ? 3 : G];  // IQ2: step j's words; IQ1_S_R4: 8 blocks' index words, then their qh halves
    };
    const auto load_group = [&](int p) {
        CodeGroup gr;
        if constexpr (IQ1) {
            gr.w[0] = load_u4(qbase + qoff + uint32_t(64 * p));
            gr.w[1] = load_u4(qbase + qoff + uint32_t(64 * p + 16));
            gr.w[2] = load_u4(hbase + hoff + uint32_t(32 * p));
        } else {
#pragma unroll
            for (int j = 0; j < G; ++j) gr.w[j] = load_u4(qbase + qoff + uint32_t(32 * G * p + 16 * j));
        }
        return gr;
    };
    // step j of a group; IQ1_S_R4: blocks 2j, 2j+1 (index words, qh halves in one word)
    const auto group_step = [](const CodeGroup &gr, int j) {
        if constexpr (IQ1) {
            const uint4_t &w = gr.w[j >> 1];
            return uint4_t{(j & 1) ? w.z : w.x, (j & 1) ? w.w : w.y, gr.w[2][j], 0u};
        } else {
            return gr.w[j];
        }
    };

    uint4_t xa[kXPer];
    constexpr std::integral_constant<int, kXPer> kAllPasses{};
    load_x(0, xa, kAllPasses);
    // IQ2_K without a dv plane in LDS: this lane's dv words, one per four steps
    const uint32_t *dvp = reinterpret_cast<const uint32_t *>(static_cast<const uint8_t *>(a.s3) + row0 * (K / 128) +
                                                             wl * uint32_t(K / 128));
    constexpr bool DV_WORDS = MEMBER == IQ2_K && !S::DV_IN_LDS;
    uint32_t dvw = DV_WORDS ? dvp[0] : 0u, dvn = 0u;
    CodeGroup grp = load_group(0), grpn{};
    store_x(0, xa, kAllPasses);
    __syncthreads();  // scale planes and the first activations are in LDS
    // row scale, applied to the sums: IQ2_KS from LDS (rows past out_features
    // read LDS junk, never stored), IQ1_S_R4 from its stream (an in-bounds
    // row); IQ2_K's are per super-block, in its pools
    _Float16 d = 0.f16;
    if constexpr (MEMBER == IQ2_KS)
        d = half_of_bits(*reinterpret_cast<const uint16_t *>(sc.dv + lrow * S::DV_S));
    else if constexpr (IQ1)
        d = half_of_bits(static_cast<const uint16_t *>(a.s2)[row0 + wl]);

    // A tile of at most 32 real slots runs the second slot block's MFMAs for
    // nothing: skip them (its slots 32 .. 63 are past the tile's end, never
    // stored, so their accumulators do not exist).
    const auto run_steps = [&](auto slot_blocks) {
        constexpr int MB = decltype(slot_blocks)::value;
        float16_t acc[MB];
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[mb][r] = 0.f;
        for (int s0 = 0; s0 < STEPS; s0 += G) {
#pragma unroll
          for (int j = 0; j < G; ++j) {
            const int s = s0 + j;
            const bool more = s + 1 < STEPS;
            if (more) load_x(s + 1, xa, slot_blocks);
            if (j == 0 && s0 + G < STEPS) grpn = load_group((s0 + G) / G);  // the next group, a group ahead
            if constexpr (DV_WORDS) {
                if ((s & 3) == 0 && s + 4 < STEPS) dvn = dvp[(s >> 2) + 1];  // the next group's word, a group ahead
            }
            Pool p[4];
            uint32_t words[4];
            uint4_t sels[IQ1 ? 4 : 1];
            if constexpr (IQ1) {
                fused_iq1(group_step(grp, j), grid, ptab, p, sels);
            } else {
                // the lane's sub-blocks are those the one-step order gives
                // step G(s/G) + kg's lane group j
                fused_pools<MEMBER, K>(sc, lrow, G * (s / G) + (G > 1 ? kg : 0), G > 1 ? j : kg, dvw, ptab, p);
                const uint4_t q = group_step(grp, j);
#pragma unroll
                for (int w = 0; w < 4; ++w) words[w] = q[w];
            }
            const uint8_t *xb = xs[s & 1] + ln * kXStride + 128 * kg;
            // A operands of MFMA u (slot blocks 0 .. MB-1)
            const auto read_a = [&](int u, half8_t *af) {
#pragma unroll
                for (int mb = 0; mb < MB; ++mb)
                    af[mb] = __builtin_bit_cast(half8_t, *reinterpret_cast<const uint4_t *>(
                                                             xb + 32 * mb * kXStride + 64 * (u >> 2) + 16 * (u & 3)));
            };
            half8_t af[MB], afn[MB];
            read_a(0, af);
            // Word w feeds MFMAs u = 2w, 2w+1 (weights 16(w%2) + 8h .. +7 of
            // sub-block 2kg + w/2, paired order); expanding word w+1 overlaps
            // word w's MFMAs.
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                uint32_t bw[8];
                if constexpr (IQ1)
                    expand_sel_paired(sels[w], p[w], bw);
                else
                    expand_word_paired(words[w], p[w], bw);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const int u = 2 * w + h;
                    if (u < 7) read_a(u + 1, afn);
                    const half8_t bf = __builtin_bit_cast(half8_t, uint4_t{bw[h], bw[2 + h], bw[4 + h], bw[6 + h]});
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb) {
                        acc[mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[mb], bf, acc[mb], 0, 0, 0);
                        af[mb] = afn[mb];
                    }
                }
            }
            if (more) store_x((s + 1) & 1, xa, slot_blocks);  // the buffer every wavefront finished reading before the last barrier
            if (j == G - 1) grp = grpn;
            if constexpr (DV_WORDS) {
                if ((s & 3) == 3) dvw = dvn;
            }
            __syncthreads();
          }
        }

        const float dscale = float(d);
        // D layout (32x32): lane l, register r holds row 8(r/4) + 4(l/32) +
        // r%4 of column l % 32.
        if (!wv) return;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t dst = slot_dst[32 * mb + 8 * (r >> 2) + 4 * kg + (r & 3)];
                if (dst != kNoStore)
                    a.y[size_t(dst & 0x7fffffffu) * a.N + n0 + lrow] =
                        (dst >> 31) ? uint16_t(float_to_half_bits(MEMBER == IQ2_K ? acc[mb][r] : acc[mb][r] * dscale))
                                    : kHalfNaN;
            }
        }
    };
    if (gend - m0 <= 32)  // uniform per block
        run_steps(std::integral_constant<int, 1>{});
    else
        run_steps(std::integral_constant<int, 2>{});
}

// ---- wide tiles -------------------------------------------------------------------

constexpr int kWideThreads = 256;
constexpr int kWideBN = 256;  // weight rows per block: 64 a wavefront

// One lane's weights of one row (ln) in steps of 128, as the 64-slot tile
// takes them, so that both sum an element in one order: lane group kg the
// sub-blocks 2kg, 2kg + 1 of a step (IQ1_S_R4, whose steps go in groups of
// four: elements 512p + 256kg + 64j .. +63 of group p in its step j).  Code
// words a step (IQ1_S_R4: two) ahead; scales of four steps at once (the IQ2
// members).
template <int MEMBER, int K>
struct WideLane {
    static constexpr bool IQ1 = MEMBER == IQ1_S_R4;
    uint4_t q;   // IQ2: a step's code words; IQ1_S_R4: two steps' index words
    uint2_t h;   // IQ1_S_R4: two steps' qh words

    __device__ __forceinline__ void load(const FewPlanes<MEMBER, K> &pl, uint32_t row, int kg, int s) {
        using P = FewPlanes<MEMBER, K>;
        if constexpr (IQ1) {
            const uint32_t p = uint32_t(s) >> 2, t = (uint32_t(s) >> 1) & 1u;  // steps 4p + 2t, 4p + 2t + 1
            q = buffer_u4(pl.p[0], row * P::ROW[0] + 32 * kg, 64 * p + 16 * t);
            h = __builtin_amdgcn_raw_buffer_load_b64(pl.p[1], row * P::ROW[1] + 16 * kg, 32 * p + 8 * t, 0);
        } else {
            q = buffer_u4(pl.p[0], row * P::ROW[0] + 16 * kg, 32 * s);
        }
    }
};

template <int MEMBER, int K>
struct WideScales {
    uint4_t sc;       // IQ2_KS: scl bytes of steps 4p .. 4p+3 (x, y); IQ2_K: scl words
    uint32_t e0, e1;  // IQ2_KS: sch, sex of super-blocks 2p, 2p+1; IQ2_K: sex of the four steps, dv

    __device__ __forceinline__ void load(const FewPlanes<MEMBER, K> &pl, uint32_t row, int p) {
        using P = FewPlanes<MEMBER, K>;
        if constexpr (MEMBER == IQ2_KS) {
            const uint2_t v = __builtin_amdgcn_raw_buffer_load_b64(pl.p[1], row * P::ROW[1], 8 * p, 0);
            sc.x = v.x;
            sc.y = v.y;
            e0 = __builtin_amdgcn_raw_buffer_load_b16(pl.p[2], row * P::ROW[2], 2 * p, 0);
            e1 = __builtin_amdgcn_raw_buffer_load_b16(pl.p[3], row * P::ROW[3], 2 * p, 0);
        } else if constexpr (MEMBER == IQ2_K) {
            sc = buffer_u4(pl.p[1], row * P::ROW[1], 16 * p);
            e0 = __builtin_amdgcn_raw_buffer_load_b32(pl.p[2], row * P::ROW[2], 4 * p, 0);
            e1 = __builtin_amdgcn_raw_buffer_load_b32(pl.p[3], row * P::ROW[3], 4 * p, 0);
        }
    }
    // the tables of step 4p + i, lane group kg
    __device__ __forceinline__ void tables(int i, int kg, const uint2_t *ptab, Pool *p) const {
        if constexpr (MEMBER == IQ2_KS) {
            const uint32_t scl = (i < 2 ? sc.x : sc.y) >> (16 * (i & 1) + 8 * kg);
            const int bit = 8 * (i >> 1) + 4 * (i & 1) + 2 * kg;
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const uint32_t e =
                    ((scl >> (4 * t)) & 15u) | (((e0 >> (bit + t)) & 1u) << 4) | (((e1 >> (bit + t)) & 1u) << 5);
                const uint2_t v = ptab[e];
                p[2 * t] = {v.x, v.y};
                p[2 * t + 1] = p[2 * t];
            }
        } else if constexpr (MEMBER == IQ2_K) {
            iq2k_pools((sc[i] >> (16 * kg)) & 0xffffu, (e0 >> (8 * i + 4 * kg)) & 15u,
                       half_of_bits((e1 >> (16 * (i >> 1))) & 0xffffu), ptab, p);
        }
    }
};

// Tiles of up to 128 slots, for calls whose experts have many: four wavefronts
// of 64 weight rows, each for all the tile's slots, so an activation fragment
// read from LDS feeds two MFMAs and a decoded weight four (the 64-slot tile's:
// one and two).  128 of a wavefront's 256 VGPRs are accumulators; two blocks a
// CU, one wavefront of each a SIMD: one's VALU work runs under the other's
// MFMAs (290 VALU a step of 64 MFMAs of 32 cycles).  The block's scales
// come straight from their planes, four steps at a time, and the activations
// (64 rows at a time, half a step ahead) are the only thing staged.  Groups
// are cut into 128-slot tiles, a last one of more than 64 slots among them;
// what is left (at most 64 slots a group) goes last in the list, so the short
// tiles fill the end of the launch.  Over the real slots of the calls listed
// at takes_wide_tiles it reaches 0.86 (many rests) to 1.08 PFLOP/s, where an
// 8192-wide fp16 library product reaches 1.08 on this card (the clock its
// power allows).  IQ2_KS's form holds 256 VGPRs and spills two; the others none.
template <int MEMBER, int K>
__global__ __launch_bounds__(kWideThreads) __attribute__((amdgpu_waves_per_eu(2, 2)))
void wide_gemm_kernel(FusedArgs a) {
    constexpr bool IQ1 = MEMBER == IQ1_S_R4;
    constexpr int STEPS = K / kFusedKS;
    static_assert(STEPS % 4 == 0, "whole groups of scales");
    __shared__ FusedScan ts;
    __shared__ uint32_t slot_dst[kWideBM];
    __shared__ uint2_t ptab[MEMBER == IQ2_K ? 32 : IQ1 ? 16 : 64];
    __shared__ __attribute__((aligned(16))) uint16_t codes[IQ1 ? IQK_IQ1S_GRID_SIZE : 8];
    __shared__ __attribute__((aligned(16))) uint8_t xs[2][kWideBM * kXStride];

    const int tid = threadIdx.x;
    const uint32_t ncb = (a.N + kWideBN - 1) / kWideBN;
    // the wide tiles first (the long ones), then the rests
    const uint32_t xcd = blockIdx.x & 7u, nth = (blockIdx.x >> 3) / ncb, cblock = (blockIdx.x >> 3) % ncb;
    const auto size_of = [&](uint32_t e) { return a.offs[e + 1] - a.offs[e]; };
    uint32_t g, mtile, share;
    if (!claim_tile<kCutWide, kWideThreads>(size_of, a.n_groups, xcd, nth, ts, g, mtile, share)) {
        if (nth < share) return;  // uniform
        __syncthreads();          // the first claim's totals have been read
        const uint32_t wide = share;
        if (!claim_tile<kCutRest, kWideThreads>(size_of, a.n_groups, xcd, nth - wide, ts, g, mtile, share)) return;
        mtile = (a.offs[g + 1] - a.offs[g]) / kWideBM;
    }
    const uint32_t gend = min(a.offs[g + 1], a.n_slots);
    const uint32_t m0 = a.offs[g] + mtile * kWideBM;
    const uint32_t n0 = cblock * kWideBN;
    const size_t row0 = size_t(g) * a.out_rows + a.row_start + n0;
    const FewPlanes<MEMBER, K> planes(a, row0);

    const int wave = tid >> 6, l = tid & 63, ln = l & 31, kg = l >> 5;
    const uint32_t wrow = uint32_t(64 * wave + ln);  // and wrow + 32
    WideLane<MEMBER, K> cur[2], nxt[2];
    WideScales<MEMBER, K> sc[2], scn[2];
#pragma unroll
    for (int b = 0; b < 2; ++b) {
        cur[b].load(planes, wrow + 32 * b, kg, 0);
        if constexpr (!IQ1) sc[b].load(planes, wrow + 32 * b, 0);
    }
    if constexpr (MEMBER == IQ2_K) {
        if (tid < 32) ptab[tid] = reinterpret_cast<const uint2_t *>(kIq2kProducts.w)[tid];
    } else if constexpr (IQ1) {
        if (tid < 16) ptab[tid] = kIq1Pools.p[tid];
        static_assert(IQK_IQ1S_GRID_SIZE == 8 * kWideThreads, "eight grid entries a thread");
        reinterpret_cast<uint4_t *>(codes)[tid] = reinterpret_cast<const uint4_t *>(iqk_iq1s_grid_codes)[tid];
    } else {
        if (tid < 64) ptab[tid] = kIq2ksPools.p[tid];
    }
    // staging: thread t moves 16-byte chunk t % 16 of slot rows t / 16 + 16 i; a
    // row past the tile's last slot, or past x, lies past x's buffer: zeros
    const int xrow = tid / kXChunks, xchunk = tid % kXChunks;
    constexpr int ROWS_A_PASS = kWideThreads / kXChunks, PASSES = int(kWideBM) / ROWS_A_PASS;
    const uint32_t xbytes = a.n_x_rows * uint32_t(2 * K);
    const __amdgpu_buffer_rsrc_t xbuf = buffer_of(a.x, xbytes);
    uint32_t xoff[PASSES];
#pragma unroll
    for (int i = 0; i < PASSES; ++i) {
        const uint32_t xp = m0 + uint32_t(xrow + ROWS_A_PASS * i);
        const bool live = xp < gend;
        const uint32_t row = live ? a.xr[xp] : a.n_x_rows;
        const bool xv = row < a.n_x_rows;  // else its output is NaN
        xoff[i] = xv ? row * uint32_t(2 * K) + uint32_t(16 * xchunk) + (IQ1 && xchunk >= 8 ? 384u : 0u) : xbytes;
        if (xchunk == 0) {
            uint32_t dst = kNoStore;
            if (live) {
                const uint32_t yrow = a.yr ? a.yr[xp] : xp;
                if (yrow < a.n_slots) dst = yrow | (xv ? 0x80000000u : 0u);
            }
            slot_dst[xrow + ROWS_A_PASS * i] = dst;
        }
    }
    constexpr int BATCH = PASSES / 2;  // rows go in two batches of 64
    const auto load_x = [&](int s, int b, uint4_t (&v)[BATCH]) {
        const uint32_t off = IQ1 ? uint32_t(1024 * (s >> 2) + 128 * (s & 3)) : uint32_t(256 * s);
#pragma unroll
        for (int i = 0; i < BATCH; ++i) v[i] = buffer_u4(xbuf, xoff[BATCH * b + i], off);
    };
    const auto store_x = [&](int buf, int b, const uint4_t (&v)[BATCH]) {
        uint8_t *dst = xs[buf] + (xrow + 64 * b) * kXStride + 16 * xchunk;
#pragma unroll
        for (int i = 0; i < BATCH; ++i)
            *reinterpret_cast<uint4_t *>(dst + ROWS_A_PASS * kXStride * i) =
                uint4_t{perm(v[i].z, v[i].x, 0x05040100u), perm(v[i].z, v[i].x, 0x07060302u),
                        perm(v[i].w, v[i].y, 0x05040100u), perm(v[i].w, v[i].y, 0x07060302u)};
    };
    uint4_t xv[BATCH];
    load_x(0, 0, xv);
    store_x(0, 0, xv);
    if (gend - m0 > uint32_t(kFusedBM)) {  // uniform
        load_x(0, 1, xv);
        store_x(0, 1, xv);
    }
    __syncthreads();

    // MB blocks of 32 slots
    const auto run = [&](auto blocks) {
        constexpr int MB = decltype(blocks)::value;

        float16_t acc[2][MB];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[b][mb][r] = 0.f;
        const uint8_t *const abase = xs[0] + ln * kXStride + 128 * kg;
        // step 4p + i, the code words in `now`, the next step's to `then`
        const auto step = [&](int p, int i, const WideLane<MEMBER, K> (&now)[2], WideLane<MEMBER, K> (&then)[2]) {
            const int s = 4 * p + i;
            const bool more = s + 1 < STEPS;
            if (more) load_x(s + 1, 0, xv);
            if (more && (!IQ1 || (i & 1))) {
#pragma unroll
                for (int b = 0; b < 2; ++b) then[b].load(planes, wrow + 32 * b, kg, s + 1);
            }
            if (!IQ1 && i == 0 && p + 1 < STEPS / 4) {
#pragma unroll
                for (int b = 0; b < 2; ++b) scn[b].load(planes, wrow + 32 * b, p + 1);
            }
            Pool pool[2][4];
            uint32_t words[2][4];
#pragma unroll
            for (int b = 0; b < 2; ++b) {
                if constexpr (IQ1) {
                    const uint32_t hw = i & 1 ? now[b].h.y : now[b].h.x;
#pragma unroll
                    for (int t = 0; t < 2; ++t) {  // blocks 2j, 2j + 1 of the two steps
                        const uint32_t qw = now[b].q[2 * (i & 1) + t], h = (hw >> (16 * t)) & 0xffffu;
                        const uint2_t v = ptab[(h >> 12) & 15u];
                        pool[b][2 * t] = {v.x, v.y};
                        pool[b][2 * t + 1] = pool[b][2 * t];
                        uint32_t c[4];
#pragma unroll
                        for (int k = 0; k < 4; ++k) c[k] = codes[((qw >> (8 * k)) & 0xffu) | (((h >> (3 * k)) & 7u) << 8)];
                        words[b][2 * t] = perm(c[1], c[0], 0x05040100u);
                        words[b][2 * t + 1] = perm(c[3], c[2], 0x05040100u);
                    }
                } else {
                    sc[b].tables(i, kg, ptab, pool[b]);
#pragma unroll
                    for (int w = 0; w < 4; ++w) words[b][w] = now[b].q[w];
                }
            }
            const uint8_t *const ab = abase + (s & 1) * int(sizeof(xs[0]));
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                uint32_t bw[2][8];
#pragma unroll
                for (int b = 0; b < 2; ++b) expand_word_paired(words[b][w], pool[b][w], bw[b]);
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    half8_t af[MB];
#pragma unroll
                    for (int mb = 0; mb < MB; ++mb)
                        af[mb] = __builtin_bit_cast(
                            half8_t, *reinterpret_cast<const uint4_t *>(ab + 32 * mb * kXStride + 32 * w + 16 * h));
#pragma unroll
                    for (int b = 0; b < 2; ++b) {
                        const half8_t bf = __builtin_bit_cast(half8_t, uint4_t{bw[b][h], bw[b][2 + h], bw[b][4 + h], bw[b][6 + h]});
#pragma unroll
                        for (int mb = 0; mb < MB; ++mb)
                            acc[b][mb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[mb], bf, acc[b][mb], 0, 0, 0);
                    }
                }
                if (w == 1 && more) {
                    store_x((s + 1) & 1, 0, xv);
                    if (MB > 2) load_x(s + 1, 1, xv);
                }
            }
            if (MB > 2 && more) store_x((s + 1) & 1, 1, xv);
            if (!IQ1 && i == 3) {
#pragma unroll
                for (int b = 0; b < 2; ++b) sc[b] = scn[b];
            }
            __syncthreads();
        };
#pragma unroll 1
        for (int p = 0; p < STEPS / 4; ++p) {
            if constexpr (IQ1) {  // a lane's words serve two steps
                step(p, 0, cur, nxt);
                step(p, 1, cur, nxt);
                step(p, 2, nxt, cur);
                step(p, 3, nxt, cur);
            } else {
                step(p, 0, cur, nxt);
                step(p, 1, nxt, cur);
                step(p, 2, cur, nxt);
                step(p, 3, nxt, cur);
            }
        }

#pragma unroll
        for (int b = 0; b < 2; ++b) {
            const uint32_t col = n0 + wrow + 32 * b;
            if (col >= a.N) continue;
            float d = 1.f;
            if constexpr (MEMBER == IQ2_KS) d = float(half_of_bits(static_cast<const uint16_t *>(a.s4)[row0 + wrow + 32 * b]));
            if constexpr (IQ1) d = float(half_of_bits(static_cast<const uint16_t *>(a.s2)[row0 + wrow + 32 * b]));
#pragma unroll
            for (int mb = 0; mb < MB; ++mb) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const uint32_t dst = slot_dst[32 * mb + 8 * (r >> 2) + 4 * kg + (r & 3)];
                    if (dst != kNoStore)
                        a.y[size_t(dst & 0x7fffffffu) * a.N + col] =
                            (dst >> 31) ? uint16_t(float_to_half_bits(MEMBER == IQ2_K ? acc[b][mb][r] : acc[b][mb][r] * d))
                                        : kHalfNaN;
                }
            }
        }
    };
    const uint32_t slots = gend - m0;
    // the empty asm keeps the forms' code apart (merged ahead of the branches
    // it costs each of them registers)
    if (slots > 96u) {
        asm volatile("" ::"n"(4));
        run(std::integral_constant<int, 4>{});
    } else if (slots > 64u) {
        asm volatile("" ::"n"(3));
        run(std::integral_constant<int, 3>{});
    } else if (slots > 32u) {
        asm volatile("" ::"n"(2));
        run(std::integral_constant<int, 2>{});
    } else {
        asm volatile("" ::"n"(1));
        run(std::integral_constant<int, 1>{});
    }
}

// Calls of many slots take the wide tiles: kWideMinSlots a group on average,
// and kWideMinWork slots x column blocks, three rounds of the 512 blocks the
// chip holds.  Measured (64-slot tiles -> wide, the kernel alone; routing
// uniform unless Zipf): IQ2_K gate, 256 experts, Zipf, 192 slots a group 1024
// -> 940 us, IQ2_KS 954 -> 926; 64 experts, 768: 844 -> 774; 32, 1536: 840 ->
// 763 (1081 TFLOP/s); IQ2_K down, 160, 230: 776 -> 719; IQ1_S_R4 gate, 128,
// Zipf, 384: 884 -> 815.  Below the line: 256 experts at 144 (a full wide
// tile and 16 more) 761 -> 807, at 48 328 -> 380; 32 experts at 192 (0.75 of a
// round) 143 -> 154.  A launch of their own for the rests measured the same or
// slower (32 experts, 192: 166; 128, Zipf, 384: 850 us).
constexpr uint64_t kWideMinSlots = 160;
constexpr uint64_t kWideMinWork = 3 * 512 * uint64_t(kWideBM);

//
// The wide tiles and the 64-slot form sum an element in one order, the
// few-slot form in another.  So a row range below the line, of an expert whose
// full rows lie above it, keeps to the 64-slot form (wide_order), and ranges
// concatenate to the full call bit for bit.  That costs a range nothing that
// shows (8192 tokens Zipf over 256 experts, IQ2_KS gate, 256 rows: 150.3 ->
// 151.3 us); wide tiles for every range of such an expert would do it too, but
// a range of few blocks then waits on its longest tile (32 experts, 2048
// tokens, down, 256 rows: 31 -> 56 us; the first one, 150 -> 166).
inline bool takes_wide_tiles(uint64_t rows, uint64_t slots, uint64_t groups) {
    static_assert(kWideBN == kFusedBN, "both forms cut the rows alike");
    const uint64_t ncb = (rows + kFusedBN - 1) / kFusedBN;
    return slots >= kWideMinSlots * groups && slots * ncb >= kWideMinWork;
}

// An upper bound on the 64-slot tiles of a call.
inline uint64_t most_tiles(uint64_t slots, uint64_t groups) {
    return std::min(slots, (slots + kFusedBM - 1) / kFusedBM + groups);
}

// Calls whose blocks route for themselves (count_pairs, list_pairs): one
// block's routing takes about 1 us where the launch it replaces took 3 to 4, so
// it pays for about three rounds of the 512 blocks the chip holds.  Measured
// (route launch -> own, us a call): 32 experts, 4 of 24 to 149 tokens, up to
// 736 blocks, IQ2_KS gate 29.5 -> 26.9, 33.6 -> 30.6, 36.1 -> 33.5, IQ1_S_R4
// down 27.1 -> 23.6, 28.9 -> 25.2, 34.4 -> 31.6; 256 experts, 6 of 12 and 24
// tokens, Zipf, 576 and 1152 blocks, gate: 44.0 -> 41.2, 49.2 -> 46.2.  Past the
// line: 96 experts, down, 1664 blocks: 68.8 -> 72.7; 256 experts, down, 4192
// blocks: IQ1_S_R4 127.9 -> 135.1.
constexpr uint64_t kSelfBlocks = 3 * 512;

inline bool takes_own_routing(uint64_t rows, uint64_t slots, uint64_t groups) {
    const uint64_t ncb = (rows + kFusedBN - 1) / kFusedBN;
    return slots <= kSelfPairs && groups <= kSelfExperts && most_tiles(slots, groups) * ncb <= kSelfBlocks &&
           !takes_wide_tiles(rows, slots, groups);
}

template <int MEMBER, int K>
int launch_fused(FusedArgs a, hipStream_t st) {
    const uint64_t ncb = (a.N + kFusedBN - 1) / kFusedBN, slots = a.n_slots, groups = a.n_groups;
    const bool wide = takes_wide_tiles(a.N, slots, groups);
    a.wide_order = takes_wide_tiles(a.out_rows, slots, groups) ? 1u : 0u;
    // tiles an XCD: of the 64-slot cut; or of the wide tiles (each of more
    // than 64 slots) and the rests (at most one a group)
    const uint64_t share = wide ? (std::min(slots / (kFusedBM + 1), slots / kWideBM + groups) + 7) / 8 +
                                      (std::min(slots, groups) + 7) / 8
                                : (most_tiles(slots, groups) + 7) / 8;
    const uint64_t blocks = 8 * share * ncb;
    if (blocks > 0x7fffffffull) return IQK_ERR_ARGUMENT;
    if (wide)
        hipLaunchKernelGGL((wide_gemm_kernel<MEMBER, K>), dim3{uint32_t(blocks)}, dim3{kWideThreads}, 0, st, a);
    else if (a.ids)
        hipLaunchKernelGGL((fused_gemm_kernel<MEMBER, K, true>), dim3{uint32_t(blocks)}, dim3{kFusedThreads}, 0, st, a);
    else
        hipLaunchKernelGGL((fused_gemm_kernel<MEMBER, K, false>), dim3{uint32_t(blocks)}, dim3{kFusedThreads}, 0, st, a);
    return record_launch(hipGetLastError());
}

// Slot lists and offsets, or (ids set) the pairs' ids.
int fused_entry(int member, int64_t in_features, int64_t out_features, int64_t num_experts,
                const void *x, int64_t n_x_rows, const void *const *streams, int n_streams, int64_t row_start,
                int64_t rows, const uint32_t *group_offsets, const uint32_t *x_rows, const uint32_t *y_rows,
                int64_t n_slots, void *y, void *stream, const void *ids, bool wide_ids, int64_t pairs_per_row) {
    if (!member_ok(member)) return IQK_ERR_MEMBER;
    if (!width_sized(in_features)) return IQK_ERR_GEOMETRY;
    if (out_features <= 0 || out_features > (int64_t(1) << 24)) return IQK_ERR_GEOMETRY;
    // 32-bit offsets within an expert's code plane (in/4 bytes a row) and x
    if (out_features * (in_features / 4) >= (int64_t(1) << 32)) return IQK_ERR_GEOMETRY;
    if (row_start < 0 || rows <= 0 || row_start + rows > out_features) return IQK_ERR_GEOMETRY;
    if (num_experts <= 0 || num_experts > (int64_t(1) << 20)) return IQK_ERR_ARGUMENT;
    if (n_slots < 0 || n_slots > (int64_t(1) << 30) || n_x_rows < 0 || n_x_rows > 0xffffffffll)
        return IQK_ERR_ARGUMENT;
    if (n_slots == 0) return IQK_OK;
    if (!x || !y || (!ids && (!group_offsets || !x_rows)) || !streams_ok(streams, n_streams, member)) return IQK_ERR_ARGUMENT;
    if (n_x_rows == 0 || n_x_rows * in_features * 2 >= (int64_t(1) << 32)) return IQK_ERR_ARGUMENT;
    FusedArgs a;
    a.x = static_cast<const uint16_t *>(x);
    a.s0 = streams[0]; a.s1 = streams[1]; a.s2 = streams[2];
    a.s3 = n_streams > 3 ? streams[3] : nullptr;
    a.s4 = n_streams > 4 ? streams[4] : nullptr;
    a.offs = group_offsets;
    a.xr = x_rows;
    a.yr = y_rows;
    a.y = static_cast<uint16_t *>(y);
    a.N = uint32_t(rows);
    a.out_rows = uint32_t(out_features);
    a.row_start = uint32_t(row_start);
    a.n_groups = uint32_t(num_experts);
    a.n_slots = uint32_t(n_slots);
    a.n_x_rows = uint32_t(n_x_rows);
    a.ids = static_cast<const uint32_t *>(ids);
    a.wide_ids = wide_ids ? 1u : 0u;
    a.pairs_per_row = uint32_t(pairs_per_row);
    hipStream_t st = as_stream(stream);
    const bool w4096 = in_features == 4096;
    switch (member) {
        case IQK_MEMBER_IQ2_KS: return w4096 ? launch_fused<IQ2_KS, 4096>(a, st) : launch_fused<IQ2_KS, 2048>(a, st);
        case IQK_MEMBER_IQ2_K: return w4096 ? launch_fused<IQ2_K, 4096>(a, st) : launch_fused<IQ2_K, 2048>(a, st);
        default: return w4096 ? launch_fused<IQ1_S_R4, 4096>(a, st) : launch_fused<IQ1_S_R4, 2048>(a, st);
    }
}

}  // namespace iqk

extern "C" {

int iqk_fused_gemm(int member, int64_t in_features, int64_t out_features, int64_t num_experts, const void *x,
                   int64_t n_x_rows, const void *const *streams, int n_streams, int64_t row_start, int64_t rows,
                   const uint32_t *group_offsets, const uint32_t *x_rows, const uint32_t *y_rows, int64_t n_slots,
                   void *y, void *stream) {
    return iqk::fused_entry(member, in_features, out_features, num_experts, x, n_x_rows, streams, n_streams, row_start,
                            rows, group_offsets, x_rows, y_rows, n_slots, y, stream, nullptr, false, 1);
}

int iqk_prefill(int member, int64_t in_features, int64_t out_features, int64_t num_experts, const void *x,
                int64_t n_x_rows, const void *const *streams, int n_streams, int64_t row_start, int64_t rows,
                const void *ids, int wide_ids, int64_t n_pairs, int64_t rows_per_pair, int64_t pairs_per_x_row,
                uint32_t *work, void *y, void *stream) {
    using namespace iqk;
    constexpr int64_t kLim = int64_t(1) << 31;
    // what the route refuses, before a product of its factors or an address of its lists is formed
    if (n_pairs < 0 || n_pairs >= kLim || rows_per_pair <= 0 || rows_per_pair >= kLim || pairs_per_x_row <= 0 ||
        pairs_per_x_row >= kLim || n_x_rows < 0 || n_x_rows >= kLim || n_pairs * rows_per_pair >= kLim)
        return IQK_ERR_ARGUMENT;
    if (n_pairs == 0) return IQK_OK;
    if (!ids || !work) return IQK_ERR_ARGUMENT;
    // every activation row a pair names lies in x
    if (((n_pairs - 1) / pairs_per_x_row + 1) * rows_per_pair > n_x_rows) return IQK_ERR_ARGUMENT;
    const int64_t slots = n_pairs * rows_per_pair;
    if (rows > 0 && num_experts > 0 && rows_per_pair == 1 &&
        takes_own_routing(uint64_t(rows), uint64_t(slots), uint64_t(num_experts)))
        return fused_entry(member, in_features, out_features, num_experts, x, n_x_rows, streams, n_streams, row_start,
                           rows, nullptr, nullptr, nullptr, slots, y, stream, ids, wide_ids != 0, pairs_per_x_row);
    uint32_t *const x_rows = work, *const y_rows = work + slots, *const offsets = work + 2 * slots;
    const int rc = wide_ids ? iqk_route_ids64(static_cast<const int64_t *>(ids), n_pairs, num_experts, rows_per_pair,
                                              pairs_per_x_row, n_x_rows, offsets, x_rows, y_rows, stream)
                            : iqk_route(static_cast<const uint32_t *>(ids), n_pairs, num_experts, rows_per_pair,
                                        pairs_per_x_row, n_x_rows, offsets, x_rows, y_rows, stream);
    if (rc != IQK_OK) return rc;
    return fused_entry(member, in_features, out_features, num_experts, x, n_x_rows, streams, n_streams, row_start, rows,
                       offsets, x_rows, y_rows, slots, y, stream, nullptr, false, 1);
}

}  // extern "C"
