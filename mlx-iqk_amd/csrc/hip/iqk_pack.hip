// ik wire -> relayout streams on the GPU (gfx950): format.pack for rows
// already in device memory.
//
// Reference: the relayout is src/mlx_iqk/format.py:478-588 (per member) and
// :612-678 (pack), done there on the CPU in numpy.  The bytes written here are
// pack's, bit for bit.
//
// A block takes whole wire rows (IQ1_S_R4: whole four-row groups), copies
// their contiguous wire bytes into LDS with 16-byte loads (a block's rows start
// 4-byte aligned: it takes an even number of rows, and every wire row is an
// even number of bytes), and then one thread per half of a 256-weight block
// (IQ1_S_R4: per 32-weight block of a group) reads its bytes from LDS and
// writes its share of every output plane; consecutive threads write consecutive
// bytes of each plane's row (the two threads of a block exchange half their
// words, so a code store covers 32 bytes a pair).
//
// Bound by the bytes in and out; what stood above that was the relayout's VALU
// work (each 2-bit field gathered by itself, 450 a block; transposed, 160), a
// thread's four 16-byte stores 64 bytes apart and dword loads.  64 experts
// [4096 x 2048], IQ2_K: 81.0 -> 60.6 us (5.26 TB/s read + written; a plain copy
// runs at 4.6), IQ2_KS 78.2 -> 59.3.  About 256 items a block: 512 took 64.7 us,
// 1024 69.7; non-temporal stores 74.4.
//
// 2-bit members: wire qs byte 32h + 16f + j (h, f in {0,1}, j < 16) carries
// in field s (bits 2s, 2s+1) the code of weight 128h + 32s + 16f + j, so
// relayout word W of a block (weights 16W .. 16W+15) gathers field
// s = (W / 2) % 4 of wire bytes 32(W / 8) + 16(W % 2) + 0..15.

#include <algorithm>

#include "iqk_device.h"
#include "iqk_host.h"

namespace iqk {

constexpr int kPackThreads = 256;
constexpr int kPackLdsBytes = 40960;
constexpr int kPackBatch = 4;  // 16-byte wire pieces a thread loads before it stores them

struct PackArgs {
    const uint8_t *wire;
    void *s0, *s1, *s2, *s3, *s4;
    uint32_t rows;       // wire rows (IQ1_S_R4: a multiple of 4)
    uint32_t row_bytes;  // ik wire bytes per row
    uint32_t nb;         // blocks per row (IQ1_S_R4: 32-weight blocks)
    uint32_t rows_per_block;
};

// `count` bytes of LDS starting at byte `off` (any alignment) as words.
__device__ __forceinline__ void lds_words(const uint8_t *lds, uint32_t off, uint32_t *out, int count_words) {
    const uint32_t *base = reinterpret_cast<const uint32_t *>(lds + (off & ~3u));
    const uint32_t sh = off & 3u;
    uint32_t prev = base[0];
    for (int i = 0; i < count_words; ++i) {
        const uint32_t next = base[i + 1];
        out[i] = __builtin_amdgcn_alignbyte(next, prev, sh);
        prev = next;
    }
}

// The 4 x 4 transpose of q's 2-bit fields: byte s of the result holds field s
// of the four bytes of q (byte k's at bits 2k, 2k+1).
__device__ __forceinline__ uint32_t transpose_fields(uint32_t q) {
    uint32_t t = (q ^ (q >> 6)) & 0x00CC00CCu;
    q ^= t ^ (t << 6);
    t = (q ^ (q >> 12)) & 0x0000F0F0u;
    return q ^ t ^ (t << 12);
}

// Fields 0 .. 3 of 16 wire bytes as relayout words: 40 VALU for four words
// (gathering each field of each dword by itself took 112).
__device__ __forceinline__ void relayout_half(const uint32_t *q, uint32_t *out) {
    uint32_t t[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) t[i] = transpose_fields(q[i]);
    const uint32_t a = perm(t[1], t[0], 0x05010400u), b = perm(t[3], t[2], 0x05010400u);  // bytes 0, 1
    const uint32_t c = perm(t[1], t[0], 0x07030602u), d = perm(t[3], t[2], 0x07030602u);  // bytes 2, 3
    out[0] = perm(b, a, 0x05040100u);
    out[1] = perm(b, a, 0x07060302u);
    out[2] = perm(d, c, 0x05040100u);
    out[3] = perm(d, c, 0x07060302u);
}

// The value of the other lane of a pair (DPP quad_perm [1,0,3,2]).
__device__ __forceinline__ uint32_t pair_swap(uint32_t v) {
    return uint32_t(__builtin_amdgcn_mov_dpp(int(v), 0xB1, 0xF, 0xF, false));
}

template <int MEMBER>
__global__ __launch_bounds__(kPackThreads) void pack_kernel(PackArgs a) {
    // the block's wire rows (+ 16 bytes, read past by lds_words): sized at
    // launch, so a CU holds as many blocks as their rows allow
    extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
    const int tid = threadIdx.x;
    const uint32_t r0 = blockIdx.x * a.rows_per_block;
    const uint32_t rows_here = min(a.rows_per_block, a.rows - r0);
    const uint64_t first = uint64_t(r0) * a.row_bytes;  // 4-byte aligned (even rows per block, even row bytes)
    const uint32_t bytes = rows_here * a.row_bytes;
    const uint32_t *src = reinterpret_cast<const uint32_t *>(a.wire + first);
    // in batches of kPackBatch 16-byte loads a thread (dword aligned), all
    // issued before any store, so the copy costs a memory latency a batch
    const uint32_t quads = bytes / 16;
    for (uint32_t i0 = 0; i0 < quads; i0 += kPackBatch * kPackThreads) {
        uint4_t v[kPackBatch];
#pragma unroll
        for (int j = 0; j < kPackBatch; ++j) {
            const uint32_t i = i0 + uint32_t(j * kPackThreads + tid);
            v[j] = load_u4(src + 4 * min(i, quads - 1u));  // past the end: re-reads the last one, never stored
        }
#pragma unroll
        for (int j = 0; j < kPackBatch; ++j) {
            const uint32_t i = i0 + uint32_t(j * kPackThreads + tid);
            if (i < quads) reinterpret_cast<uint4_t *>(lds)[i] = v[j];
        }
    }
    if (tid < int(bytes / 4 - 4 * quads)) reinterpret_cast<uint32_t *>(lds)[4 * quads + tid] = src[4 * quads + tid];
    if ((bytes & 3u) && tid == 0)  // an odd last row leaves one 16-bit unit
        *reinterpret_cast<uint16_t *>(lds + (bytes & ~3u)) = *reinterpret_cast<const uint16_t *>(a.wire + first + (bytes & ~3u));
    __syncthreads();

    if constexpr (MEMBER == IQ2_KS || MEMBER == IQ2_K) {
        // an item is half a block: 32 wire qs bytes, 8 relayout words.  Lanes
        // go in pairs (whole blocks), so every lane of a pair has an item.
        const uint32_t items = 2 * rows_here * a.nb;
        for (uint32_t it = tid; it < items; it += kPackThreads) {
            const uint32_t rl = it / (2 * a.nb), b = (it >> 1) - rl * a.nb, half = it & 1u;
            const uint64_t row = r0 + rl;
            const uint32_t rbase = rl * a.row_bytes;
            uint32_t q[8];
            if constexpr (MEMBER == IQ2_KS) {  // [d f16] then blocks [extra u16, scales[4], qs[64]]
                const uint32_t off = rbase + 2 + 70 * b;
                lds_words(lds, off + 6 + 32 * half, q, 8);
                if (half == 0) {
                    uint32_t hdr[2];
                    lds_words(lds, off, hdr, 2);
                    static_cast<uint8_t *>(a.s3)[row * a.nb + b] = uint8_t(hdr[0]);        // sex: extra low byte
                    static_cast<uint8_t *>(a.s2)[row * a.nb + b] = uint8_t(hdr[0] >> 8);   // sch: extra high byte
                    static_cast<uint32_t *>(a.s1)[row * a.nb + b] = __builtin_amdgcn_alignbyte(hdr[1], hdr[0], 2);  // scales[4]
                    if (b == 0) static_cast<uint16_t *>(a.s4)[row] = *reinterpret_cast<const uint16_t *>(lds + rbase);
                }
            } else {  // blocks [d f16, extra u16, scales[8], qs[64]]: dword aligned
                const uint32_t *blk = reinterpret_cast<const uint32_t *>(lds + rbase + 76 * b);
#pragma unroll
                for (int i = 0; i < 8; ++i) q[i] = blk[3 + 8 * half + i];
                if (half == 0) {
                    const uint32_t hdr = blk[0];
                    static_cast<uint16_t *>(a.s3)[row * a.nb + b] = uint16_t(hdr);            // dv
                    static_cast<uint16_t *>(a.s2)[row * a.nb + b] = uint16_t(hdr >> 16);      // sex, 2 bytes (LE)
                    uint32_t *scl = reinterpret_cast<uint32_t *>(static_cast<uint8_t *>(a.s1) + (row * a.nb + b) * 8);
                    scl[0] = blk[1];
                    scl[1] = blk[2];
                }
            }
            // words 2s + f of the half: field s of its bytes 16f .. 16f + 15
            uint32_t w0[4], w1[4];
            relayout_half(q, w0);
            relayout_half(q + 4, w1);
            // The pair's 64 bytes, lane by lane: each store instruction writes
            // 32 contiguous bytes a pair, the first one the even lane's half.
            uint32_t keep[4], send[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint32_t lo = i & 1 ? w1[i >> 1] : w0[i >> 1];          // words 0 .. 3 of the half
                const uint32_t hi = i & 1 ? w1[2 + (i >> 1)] : w0[2 + (i >> 1)];  // words 4 .. 7
                keep[i] = half ? hi : lo;
                send[i] = pair_swap(half ? lo : hi);
            }
            uint4_t *qs = reinterpret_cast<uint4_t *>(static_cast<uint32_t *>(a.s0) + (row * a.nb + b) * 16);
            const uint4_t own = {keep[0], keep[1], keep[2], keep[3]}, other = {send[0], send[1], send[2], send[3]};
            qs[half] = half ? other : own;      // even half: words 0 .. 3 | 4 .. 7
            qs[2 + half] = half ? own : other;  // odd half
        }
    } else {  // IQ1_S_R4: groups [d f16 x4] then blocks [qs[16] (byte 4t + k: row k), qh u16 x4]
        const uint32_t gbytes = 4 * a.row_bytes;
        const uint32_t items = (rows_here / 4) * a.nb;
        for (uint32_t it = tid; it < items; it += kPackThreads) {
            const uint32_t gl = it / a.nb, b = it - gl * a.nb;
            const uint64_t row = r0 + 4 * gl;  // first row of the group
            const uint32_t gbase = gl * gbytes;
            const uint32_t *blk = reinterpret_cast<const uint32_t *>(lds + gbase + 8 + 24 * b);  // 4-byte aligned
            const uint32_t q0 = blk[0], q1 = blk[1], q2 = blk[2], q3 = blk[3];
            const uint32_t t01 = perm(q1, q0, 0x05010400u), t23 = perm(q3, q2, 0x05010400u);  // bytes 0, 1
            const uint32_t u01 = perm(q1, q0, 0x07030602u), u23 = perm(q3, q2, 0x07030602u);  // bytes 2, 3
            const uint32_t rq[4] = {perm(t23, t01, 0x05040100u), perm(t23, t01, 0x07060302u),
                                    perm(u23, u01, 0x05040100u), perm(u23, u01, 0x07060302u)};
            const uint32_t h01 = blk[4], h23 = blk[5];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                static_cast<uint32_t *>(a.s0)[(row + k) * a.nb + b] = rq[k];
                static_cast<uint16_t *>(a.s1)[(row + k) * a.nb + b] = uint16_t((k < 2 ? h01 : h23) >> (16 * (k & 1)));
            }
            if (b == 0) {
                const uint32_t *dv = reinterpret_cast<const uint32_t *>(lds + gbase);
#pragma unroll
                for (int k = 0; k < 4; ++k)
                    static_cast<uint16_t *>(a.s2)[row + k] = uint16_t(dv[k >> 1] >> (16 * (k & 1)));
            }
        }
    }
}

}  // namespace iqk

extern "C" int iqk_pack(int member, int64_t in_features, int64_t rows, const void *wire, void *const *streams,
                        int n_streams, void *stream) {
    using namespace iqk;
    if (!member_ok(member)) return IQK_ERR_MEMBER;
    const bool iq1 = member == IQK_MEMBER_IQ1_S_R4;
    const int64_t block = iq1 ? 32 : 256;
    if (in_features <= 0 || in_features % block || in_features > (int64_t(1) << 20)) return IQK_ERR_GEOMETRY;
    if (rows < 0 || rows > 0xffffffffll || (iq1 && rows % 4)) return IQK_ERR_GEOMETRY;
    if (rows == 0) return IQK_OK;
    if (!wire || !streams || n_streams != stream_count(member)) return IQK_ERR_ARGUMENT;
    for (int i = 0; i < n_streams; ++i)
        if (!streams[i]) return IQK_ERR_ARGUMENT;
    // the kernel reads the wire as dwords and writes code words 16 bytes at a time
    if (reinterpret_cast<uintptr_t>(wire) % 4 || reinterpret_cast<uintptr_t>(streams[0]) % 16) return IQK_ERR_ARGUMENT;
    for (int i = 1; i < n_streams; ++i)
        if (reinterpret_cast<uintptr_t>(streams[i]) % 4) return IQK_ERR_ARGUMENT;
    const int64_t nb = in_features / block;
    const int64_t row_bytes = member == IQK_MEMBER_IQ2_KS ? 2 + 70 * nb : member == IQK_MEMBER_IQ2_K ? 76 * nb : 2 + 6 * nb;
    if (rows * row_bytes > (int64_t(1) << 40)) return IQK_ERR_ARGUMENT;
    // rows per block: an even number (a multiple of 4 for IQ1_S_R4) whose bytes fit the LDS copy,
    // about 256 work items per block
    const int64_t unit = iq1 ? 4 : 2;
    const int64_t per_unit_items = iq1 ? nb : 4 * nb;
    int64_t units = std::max<int64_t>(1, kPackThreads / per_unit_items);
    units = std::min<int64_t>(units, kPackLdsBytes / (unit * row_bytes));
    if (units < 1) return IQK_ERR_GEOMETRY;  // one row group does not fit the LDS copy
    PackArgs a;
    a.wire = static_cast<const uint8_t *>(wire);
    a.s0 = streams[0]; a.s1 = streams[1]; a.s2 = streams[2];
    a.s3 = n_streams > 3 ? streams[3] : nullptr;
    a.s4 = n_streams > 4 ? streams[4] : nullptr;
    a.rows = uint32_t(rows);
    a.row_bytes = uint32_t(row_bytes);
    a.nb = uint32_t(nb);
    a.rows_per_block = uint32_t(units * unit);
    const dim3 grid{uint32_t((rows + a.rows_per_block - 1) / a.rows_per_block)}, blk{kPackThreads};
    const size_t lds = (size_t(a.rows_per_block) * a.row_bytes + 16 + 15) / 16 * 16;
    hipStream_t st = as_stream(stream);
    switch (member) {
        case IQK_MEMBER_IQ2_KS: hipLaunchKernelGGL(pack_kernel<IQ2_KS>, grid, blk, lds, st, a); break;
        case IQK_MEMBER_IQ2_K: hipLaunchKernelGGL(pack_kernel<IQ2_K>, grid, blk, lds, st, a); break;
        default: hipLaunchKernelGGL(pack_kernel<IQ1_S_R4>, grid, blk, lds, st, a); break;
    }
    return record_launch(hipGetLastError());
}
