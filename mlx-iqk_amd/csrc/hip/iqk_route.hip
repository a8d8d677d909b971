// The prefill route's pair grouping on the device: token-expert pairs ->
// expert-sorted slots, in one launch.
//
// Reference: the sorted prefill hands mx.gather_mm pairs sorted by expert
// (mlx_lm's _gather_sort, src/mlx_iqk/nn.py:221-238, sorted_indices=True)
// and gather_mm groups them by rhs index.  Here the grouping is one kernel
// whose outputs are exactly what the prefill kernels take: group offsets in
// slots, and each slot's activation row and output row.
//
// A pair's key is its expert id; an id >= num_experts keys as expert 0 (its
// slots keep an activation row past x, so the prefill kernels answer them with
// NaN rows and read nothing).  Expert e's slots are
//   [#{pairs keyed below e}, #{pairs keyed below e + 1}),
// its pairs in pair order (a stable counting sort).
//
// One workgroup per expert, so a launch spreads over the chip; no workspace.
// Its wavefronts each take a contiguous share of the pairs and hold their keys
// in registers, two a register, a lane eight consecutive pairs of a piece of
// 512 (read again from L2 only past 4096 pairs a wavefront):
//   1. each lane counts its pairs keyed below e and keyed e, two at a time on
//      packed 16-bit operations;
//   2. the totals through LDS give the group offset and each wavefront's first
//      slot (the offset + the e-pairs of the wavefronts before it);
//   3. each wavefront with e-pairs writes them in order, a pair's slot being
//      its wavefront's next slot + its rank in the piece, from eight ballots.
// Every block runs over the whole id list, and with many pairs its VALU and
// SALU work on them bounds the time: with a lane's pairs 64 apart, a ballot
// pair per 64 of them (24 instructions) and the rank from each, 49152 pairs
// over 256 experts took 18.8 us, over 32 experts 24.8 and 12288 over 256 took
// 7.4; now 11.5, 12.2 and 5.9, and with 64-bit ids, whose list is twice as
// long, 15.2, 16.1 and 6.8.  Up to 2048 pairs it is latency: four wavefronts of
// one piece each take 3.2 us at 144 pairs with either ids (eight wavefronts of
// 32 ballot steps whatever their share: 5.5).  (Medians of 30 dispatches in a
// kernel trace, 32-bit ids where not said.)

#include "iqk_device.h"
#include "iqk_host.h"

namespace iqk {

constexpr int kRouteMaxExperts = 4096;
constexpr uint32_t kRouteSmall = 2048;   // pairs the small form takes
constexpr uint32_t kPiece = 512;         // pairs of a piece, eight a lane
constexpr uint32_t kPastEnd = 0xfffeu;   // the key of no pair: neither below nor an expert

struct RouteArgs {
    const uint32_t *ids;
    uint32_t *offs;
    uint32_t *xr;
    uint32_t *yr;
    uint32_t P, E, M, ppx, n_x_rows;
    uint32_t inv_ppx;  // floor(2^32 / ppx), 2^32 - 1 for ppx = 1
};

typedef unsigned short ushort2_t __attribute__((ext_vector_type(2)));

// One 32-bit id of pair p, or what a 64-bit one past 32 bits reads as: no expert.
template <bool WIDE>
__device__ __forceinline__ uint32_t load_id(const uint32_t *ids, uint32_t p) {
    if constexpr (WIDE) {
        const uint2_t id = reinterpret_cast<const uint2_t *>(ids)[p];
        return id.y ? 0xffffffffu : id.x;
    } else {
        return ids[p];
    }
}

// WIDE: 64-bit ids.  WAVES wavefronts, each holding PIECES pieces of keys.
template <bool WIDE, int WAVES, int PIECES>
__global__ __launch_bounds__(64 * WAVES) void route_kernel(RouteArgs a) {
    constexpr uint32_t ROUND = kPiece * PIECES;  // pairs a wavefront holds
    __shared__ uint32_t tot[2][WAVES];           // per wavefront: pairs keyed below e, keyed e
    const uint32_t e = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // wavefront w takes pairs [lo, hi): contiguous whole pieces, in wavefront order
    const uint32_t share = (a.P + kPiece * WAVES - 1u) / (kPiece * WAVES) * kPiece;
    const uint32_t lo = min(a.P, uint32_t(wave) * share), hi = min(a.P, lo + share);

    // The keys of pairs base + 512 t + 8 lane + k (t < PIECES, k < 8): their
    // experts, 0 for an id beyond the stack, kPastEnd past hi.  Only called
    // with lo <= base < hi.
    uint32_t keys[PIECES][4];
    const auto load = [&](uint32_t base) {
        uint32_t raw[PIECES][8];
#pragma unroll
        for (int t = 0; t < PIECES; ++t) {  // whole pieces: 16-byte loads (dword aligned, as ids are)
            if (base + kPiece * uint32_t(t + 1) <= hi) {
                const uint32_t *const ids = a.ids + ((size_t(base) + kPiece * uint32_t(t)) << (WIDE ? 1 : 0));
                if constexpr (WIDE) {
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const uint4_t v = load_u4(ids + 16 * lane + 4 * k);
                        raw[t][2 * k] = v.y ? 0xffffffffu : v.x;
                        raw[t][2 * k + 1] = v.w ? 0xffffffffu : v.z;
                    }
                } else {
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        const uint4_t v = load_u4(ids + 8 * lane + 4 * k);
#pragma unroll
                        for (int i = 0; i < 4; ++i) raw[t][4 * k + i] = v[i];
                    }
                }
            } else if (base + kPiece * uint32_t(t) < hi) {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    raw[t][k] = load_id<WIDE>(a.ids, min(base + kPiece * uint32_t(t) + uint32_t(8 * lane + k), hi - 1u));
            }
        }
#pragma unroll
        for (int t = 0; t < PIECES; ++t) {
            const uint32_t p0 = base + kPiece * uint32_t(t);
            if (p0 >= hi) {
#pragma unroll
                for (int k = 0; k < 4; ++k) keys[t][k] = kPastEnd * 0x10001u;
                continue;
            }
            uint32_t key[8];
#pragma unroll
            for (int k = 0; k < 8; ++k) key[k] = raw[t][k] < a.E ? raw[t][k] : 0u;
            if (p0 + kPiece > hi) {
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    if (p0 + uint32_t(8 * lane + k) >= hi) key[k] = kPastEnd;
            }
#pragma unroll
            for (int k = 0; k < 4; ++k) keys[t][k] = perm(key[2 * k + 1], key[2 * k], 0x05040100u);
        }
    };

    const ushort2_t ee = {static_cast<unsigned short>(e), static_cast<unsigned short>(e)}, one = {1, 1};
    uint32_t lt = 0, eq = 0;
    for (uint32_t base = lo; base < hi; base += ROUND) {
        load(base);
        ushort2_t lt2 = {0, 0}, ne2 = {0, 0};  // a lane's counts of its even and odd pairs
        uint32_t pairs = 0;
#pragma unroll
        for (int t = 0; t < PIECES; ++t) {
            if (base + kPiece * uint32_t(t) >= hi) continue;  // uniform
            pairs += 8;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const ushort2_t key = __builtin_bit_cast(ushort2_t, keys[t][k]);
                lt2 += __builtin_elementwise_min(__builtin_elementwise_sub_sat(ee, key), one);
                ne2 += __builtin_elementwise_min(key ^ ee, one);
            }
        }
        lt += uint32_t(lt2.x) + uint32_t(lt2.y);
        eq += pairs - (uint32_t(ne2.x) + uint32_t(ne2.y));
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        lt += __shfl_xor(lt, off, 64);
        eq += __shfl_xor(eq, off, 64);
    }
    if (lane == 0) {
        tot[0][wave] = lt;
        tot[1][wave] = eq;
    }
    __syncthreads();
    uint32_t first = 0, slot = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
        first += tot[0][w];
        if (w < wave) slot += tot[1][w];
    }
    slot = __builtin_amdgcn_readfirstlane(slot + first);
    if (threadIdx.x == 0) {
        a.offs[e] = first * a.M;
        if (e == a.E - 1u) a.offs[a.E] = a.P * a.M;
    }
    if (__builtin_amdgcn_readfirstlane(eq) == 0) return;  // no e-pairs in this wavefront's share

    for (uint32_t base = lo; base < hi; base += ROUND) {
        if (hi - lo > ROUND) load(base);  // one round: the keys are still held
#pragma unroll
        for (int t = 0; t < PIECES; ++t) {
            const uint32_t p0 = base + kPiece * uint32_t(t);
            if (p0 >= hi) continue;  // uniform
            uint32_t mine = 0;       // bit k: pair 8 lane + k of the piece
#pragma unroll
            for (int k = 0; k < 8; ++k)
                mine |= ((k & 1 ? keys[t][k / 2] >> 16 : keys[t][k / 2] & 0xffffu) == e ? 1u : 0u) << k;
            if (__ballot(mine != 0) == 0) continue;  // uniform
            // rank: e-pairs of the lanes before, then the lane's own in order
            uint32_t rank = 0, count = 0;
#pragma unroll
            for (int k = 0; k < 8; ++k) {
                const uint64_t m = __ballot((mine >> k) & 1u);
                rank = __builtin_amdgcn_mbcnt_hi(uint32_t(m >> 32), __builtin_amdgcn_mbcnt_lo(uint32_t(m), rank));
                count += uint32_t(__popcll(m));
            }
            while (mine) {
                const uint32_t p = p0 + 8u * uint32_t(lane) + uint32_t(__ffs(mine) - 1);
                mine &= mine - 1u;
                const uint32_t at = (slot + rank++) * a.M;
                // p / ppx: the product is short by at most one
                uint32_t q = __umulhi(p, a.inv_ppx);
                if (p - q * a.ppx >= a.ppx) ++q;
                // expert 0 also holds the ids beyond the stack
                const bool valid = e != 0 || load_id<WIDE>(a.ids, p) < a.E;
                for (uint32_t r = 0; r < a.M; ++r) {
                    a.yr[at + r] = p * a.M + r;
                    a.xr[at + r] = valid ? q * a.M + r : a.n_x_rows;
                }
            }
            slot += count;
        }
    }
}

template <bool WIDE>
int route_entry(const void *ids, int64_t n_pairs, int64_t num_experts, int64_t rows_per_pair, int64_t pairs_per_x_row,
                int64_t n_x_rows, uint32_t *group_offsets, uint32_t *x_rows, uint32_t *y_rows, void *stream) {
    if (num_experts <= 0 || num_experts > kRouteMaxExperts) return IQK_ERR_ARGUMENT;
    if (n_pairs < 0 || rows_per_pair <= 0 || pairs_per_x_row <= 0 || n_x_rows < 0) return IQK_ERR_ARGUMENT;
    // each factor bounded first, so the products below cannot overflow
    constexpr int64_t kLim = int64_t(1) << 31;
    if (n_pairs >= kLim || rows_per_pair >= kLim || pairs_per_x_row >= kLim || n_x_rows >= kLim)
        return IQK_ERR_ARGUMENT;
    if (n_pairs * rows_per_pair >= kLim) return IQK_ERR_ARGUMENT;
    if (!group_offsets || (n_pairs && (!ids || !x_rows || !y_rows))) return IQK_ERR_ARGUMENT;
    // every activation row a valid pair names lies in x
    if (n_pairs && ((n_pairs - 1) / pairs_per_x_row + 1) * rows_per_pair > n_x_rows) return IQK_ERR_ARGUMENT;
    RouteArgs a;
    a.ids = static_cast<const uint32_t *>(ids);
    a.offs = group_offsets;
    a.xr = x_rows;
    a.yr = y_rows;
    a.P = uint32_t(n_pairs);
    a.E = uint32_t(num_experts);
    a.M = uint32_t(rows_per_pair);
    a.ppx = uint32_t(pairs_per_x_row);
    a.n_x_rows = uint32_t(n_x_rows);
    a.inv_ppx = a.ppx == 1 ? 0xffffffffu : uint32_t((uint64_t(1) << 32) / a.ppx);
    const dim3 grid{uint32_t(num_experts)};
    if (a.P <= kRouteSmall)
        hipLaunchKernelGGL((route_kernel<WIDE, 4, 1>), grid, dim3{256}, 0, as_stream(stream), a);
    else
        hipLaunchKernelGGL((route_kernel<WIDE, 16, 8>), grid, dim3{1024}, 0, as_stream(stream), a);
    return record_launch(hipGetLastError());
}

}  // namespace iqk

extern "C" {

int iqk_route(const uint32_t *ids, int64_t n_pairs, int64_t num_experts, int64_t rows_per_pair,
              int64_t pairs_per_x_row, int64_t n_x_rows, uint32_t *group_offsets, uint32_t *x_rows, uint32_t *y_rows,
              void *stream) {
    return iqk::route_entry<false>(ids, n_pairs, num_experts, rows_per_pair, pairs_per_x_row, n_x_rows, group_offsets,
                                   x_rows, y_rows, stream);
}

int iqk_route_ids64(const int64_t *ids, int64_t n_pairs, int64_t num_experts, int64_t rows_per_pair,
                    int64_t pairs_per_x_row, int64_t n_x_rows, uint32_t *group_offsets, uint32_t *x_rows,
                    uint32_t *y_rows, void *stream) {
    return iqk::route_entry<true>(ids, n_pairs, num_experts, rows_per_pair, pairs_per_x_row, n_x_rows, group_offsets,
                                  x_rows, y_rows, stream);
}

}  // extern "C"
