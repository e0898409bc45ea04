// Transforms whose columns (or LDE blocks) fit one work-group's LDS, in one
// launch: source, every stage, bit reversal, scaling and store.
//
// A tile of 2^LT words holds whole blocks of 2^L, and for natural order
// output whole columns of 2^lg = 2^(L + rate).  Each of its 2^(LT - LE) lanes
// keeps 2^LE words and runs LE stages a round on them, the first on the loaded
// words; one LDS exchange between rounds.  The last round (stages below LE,
// small roots as shifts) leaves its words in LDS where they belong, so the
// stores are runs.
//
// Split.  Up to 2^12: 1024 lanes of four words (LE = 2), so that a lone small
// transform, which is one tile's latency, has four waves on each SIMD of its
// CUs rather than one, and a quarter of the serial work a lane.  2^13: eight
// words, 66 KB, still two work-groups per CU.  2^14: sixteen, one per CU.
// L and the direction are template parameters: all twiddles of a lane are
// loaded with its words.
//
// Bound up to 2^12 by the call itself (launch and wait, 15 of its 16-20 us),
// above by one tile's latency, in large batches by HBM.  Against one launch
// per pass and one for the bit reversal, same GPU, us a call: inverse of 101 x
// 2^13 39 -> 27, 400 x 2^12 44 -> 27, 400 x 2^14 98 -> 71, 20 x 2^10 25 -> 18;
// LDE of 135 x 2^13 rate 1 58 -> 41; the LDE of a commit of 20 x 2^10 rate 1
// (DIF order) 17 -> 9.
#pragma once
#include "ntt_lanes.h"

namespace zkx {

template <int LT, int LE>
struct ColumnShape {
    static constexpr int kLanes = 1 << (LT - LE), kWords = 1 << LE;
    static constexpr int kSlots = (1 << LT) + (1 << LT) / 32;
};

// Word e of lane t in a round whose register bits start at bit RB of the
// tile position.
template <int LE>
__device__ __forceinline__ uint32_t column_pos(uint32_t t, int rb, int e)
{
    return ((t >> rb) << (rb + LE)) | ((uint32_t)e << rb) | (t & ((1u << rb) - 1));
}

// A stage on 2^LE registers (reg_stage for any register count).
template <int LE, class A, class W>
__device__ __forceinline__ void column_stage(A &ar, uint64_t (&x)[1 << LE], int b, W &&w)
{
#pragma unroll
    for (int k = 0; k < (1 << LE) / 2; k += 2) {
        const int e0 = ((k >> b) << (b + 1)) | (k & ((1 << b) - 1));
        const int e1 = (((k + 1) >> b) << (b + 1)) | ((k + 1) & ((1 << b) - 1));
        ar.add_sub2(x[e0], x[e0 | (1 << b)], x[e1], x[e1 | (1 << b)]);
        ar.mul2(x[e0 | (1 << b)], w(e0), x[e1 | (1 << b)], w(e1));
    }
}

// Stages REM-1..0, the words of the first of these rounds in x; the last
// leaves the tile in x at register bit 0.
template <int LE, int REM, bool INV, class A>
__device__ __forceinline__ void column_rounds(A &ar, uint64_t *lds, uint64_t (&x)[1 << LE], const NttPass &a, uint32_t t)
{
    if constexpr (REM > LE) {
        constexpr int B0 = REM - LE;
        const uint32_t lo = t & ((1u << B0) - 1);
#pragma unroll
        for (int dd = LE - 1; dd >= 0; dd--) {
            const uint32_t mask = (2u << (B0 + dd)) - 1;
            const gptr<const uint64_t> tab = gmem(cmem(a.tw_lg)[B0 + dd + 1]);
            uint64_t w[1 << (LE - 1)];
#pragma unroll
            for (int v = 0; v < (1 << dd); v++) {
                const uint32_t k = lo | ((uint32_t)v << B0);
                w[v] = tab[INV ? (0u - k) & mask : k];
            }
            column_stage<LE>(ar, x, dd, [&](int e) { return w[e & ((1 << dd) - 1)]; });
        }
        constexpr int NEXT = B0 > LE ? B0 - LE : 0;
#pragma unroll
        for (int e = 0; e < (1 << LE); e++) lds[lds_slot(column_pos<LE>(t, B0, e))] = x[e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < (1 << LE); e++) x[e] = lds[lds_slot(column_pos<LE>(t, NEXT, e))];
        column_rounds<LE, B0, INV>(ar, lds, x, a, t);
    } else if constexpr (REM > 0) {
        last_stages<REM - 1, INV, 1 << LE>(ar, x);
    }
}

template <int LT, int LE, int L, bool INV, class A>
__device__ __forceinline__ void column_transform(A &ar, uint64_t *lds, const NttPass &a, const ColumnPost &post,
                                                 uint64_t tile, uint32_t t)
{
    constexpr int E = 1 << LE, RB = L > LE ? L - LE : 0;
    uint64_t x[E], f[E];
    // words past the end of a last, partial tile read the last word
    auto index = [&](int e) {
        const uint64_t idx = (tile << LT) + column_pos<LE>(t, RB, e);
        return idx < a.total ? idx : a.total - 1;
    };
    if (a.mode == kSrcLde) {
#pragma unroll
        for (int e = 0; e < E; e++) {
            const uint64_t idx = index(e);
            x[e] = gmem(a.src)[((idx >> (L + a.rate)) << L) + (idx & ((1ull << L) - 1))];
            f[e] = gmem(a.coset)[idx & ((1ull << (L + a.rate)) - 1)];
        }
    } else {
#pragma unroll
        for (int e = 0; e < E; e++) x[e] = A::load(gmem(a.buf)[index(e)]);
        if (!INV && a.mode == kSrcCoset) {
#pragma unroll
            for (int e = 0; e < E; e++) f[e] = gmem(a.coset)[index(e) & ((1ull << L) - 1)];
        }
    }
    if (a.mode != kSrcInPlace) {
#pragma unroll
        for (int e = 0; e < E; e += 2) ar.mul2(x[e], f[e], x[e + 1], f[e + 1]);
    }
    column_rounds<LE, L, INV>(ar, lds, x, a, t);
    // the last round's positions are its lane's own: t << LE | e
    const uint32_t shift = 32 - post.lg, mask = (uint32_t)((1ull << post.lg) - 1), first = t << LE;
    const uint32_t r0 = __builtin_bitreverse32(first);
    uint32_t to[E];
#pragma unroll
    for (int e = 0; e < E; e++)
        to[e] = post.natural ? ((first | e) & ~mask) | ((r0 | __builtin_bitreverse32((uint32_t)e)) >> shift) : first | e;
    if constexpr (INV) {
#pragma unroll
        for (int e = 0; e < E; e += 2) ar.mul2(x[e], post.scale, x[e + 1], post.scale);
        if (post.coset) {
#pragma unroll
            for (int e = 0; e < E; e += 2)
                ar.mul2(x[e], gmem(post.coset)[to[e] & mask], x[e + 1], gmem(post.coset)[to[e + 1] & mask]);
        }
    }
    // (a lane's words go to other lanes' slots: all have been read)
    if constexpr (L > LE) __syncthreads();
#pragma unroll
    for (int e = 0; e < E; e++) lds[lds_slot(to[e])] = A::result(x[e]);
}

template <int LT, int LE, int L, bool INV>
__global__ void __launch_bounds__(1 << (LT - LE)) __attribute__((amdgpu_waves_per_eu(LE < 4 ? 8 : 4)))
k_ntt_columns(const NttPass *__restrict__ passes, uint32_t npasses, NttPass one, ColumnPost post, uint64_t first)
{
    constexpr int N = ColumnShape<LT, LE>::kLanes;
    __shared__ uint64_t lds[ColumnShape<LT, LE>::kSlots];
    const uint32_t t = threadIdx.x;
    const uint64_t b = first + blockIdx.x;
    const NttPass a = pass_at(passes, npasses, one, b);
    const uint64_t tile = b - a.tile_begin;
    Lazy lazy;
    column_transform<LT, LE, L, INV>(lazy, lds, a, post, tile, t);
    __syncthreads();
    const uint64_t base = (tile << LT) + t;
    const gptr<uint64_t> p = gmem(a.buf) + base;
#pragma unroll
    for (int i = 0; i < (1 << LE); i++)
        if (base + (uint64_t)N * i < a.total) p[N * i] = lds[lds_slot(t + N * i)];
}

}  // namespace zkx
