// Natural-order transforms of 2^15 to 2^20 points in two launches, through a
// scratch buffer: the top M1 stages (k_ntt_first), then the M2 low ones with the
// bit reversal in their stores (k_ntt_second).
//
// Both work on tiles of 2^13 words, 1024 lanes of eight (66 KB of LDS, two
// work-groups per CU), as ntt_columns.h does.  Position u of a tile:
//   first   u = (j << C | q): butterfly index j (M1 bits) at stride 2^M2, 2^C
//           consecutive columns q of the stride, C = 13 - M1;
//   second  u = (x << M2 | j): 2^C rows of 2^M2 consecutive words, C = 13 - M2,
//           which differ in the top C bits of the row number, so that the
//           output of one j, reversed, is a run of 2^C words.
// A transform in place cannot store into the order it reads in, hence the
// scratch, which holds the columns of one chunk; chunks of up to 128 MiB stay
// in the last-level cache between the two launches.
//
// With 64-byte runs (M = 10) the work-groups that share 128-byte lines are
// given to one XCD (its L2 merges their halves): work-groups go to the XCDs in
// turn, so b and b + 8 take adjacent tiles.
//
// Bound: a tile's latency (two work-groups per CU hide half of it): a launch
// over 16 columns of 2^20 (268 MB of traffic) 92 and 78 us, where HBM takes 55
// and the instructions 50.  Against a strided and a contiguous pass in place
// and a bit reversal, same GPU, us a call: 64 x 2^20 846 -> 636, 256 x 2^18 774
// -> 521, 64 x 2^17 108 -> 80, LDE of 135 x 2^15 rate 3 416 -> 290, of 2 x 2^19
// rate 1 53 -> 40.
#pragma once
#include "ntt_columns.h"

namespace zkx {

constexpr int kTwoTile = 13, kTwoWords = 3;  // log2 words of a tile, and of a lane
constexpr int kTwoLanes = 1 << (kTwoTile - kTwoWords);
using TwoShape = ColumnShape<kTwoTile, kTwoWords>;

template <int C>
__device__ __forceinline__ uint64_t two_tile(uint64_t b)
{
    if constexpr (C > 3) return b;
    else return (b & ~15ull) | ((b & 7) << 1) | ((b >> 3) & 1);
}

// Word u of a first tile in its block (of 2^(M1 + s) words).
template <int M1>
__device__ __forceinline__ uint32_t first_pos(uint32_t s, uint32_t ch, uint32_t u)
{
    constexpr int C = kTwoTile - M1;
    return ((u >> C) << s) + (ch << C) + (u & ((1u << C) - 1));
}

// A stage whose twiddle for element e is b * w_{2^(DD+1)}^v, v = e mod 2^DD: the
// root is a power of two, so its other twiddles are b shifted (2^96 = -1: the
// difference taken the other way round) instead of loaded: 10 loads a lane
// instead of 22 for ten stages, whose waits and cache misses took longer than
// the shifts (64 x 2^20: 107 -> 92 us a first launch over 16 columns, 81 -> 78 a
// second).  The transforms of ntt_columns.h, whose tables stay in the first
// caches, are 1-4% slower that way.
template <int DD, bool INV, int E, class A>
__device__ __forceinline__ void root_stage(A &ar, uint64_t (&x)[E], uint64_t b)
{
    uint64_t w[1 << DD];
    static_for<0, 1 << DD>([&](auto vc) {
        constexpr int v = decltype(vc)::value;
        w[v] = ar.template shift<small_root_log<DD, v, INV>() % 96>(b);
    });
    static_for<0, E / 4>([&](auto kc) {
        constexpr int k = 2 * decltype(kc)::value;
        constexpr int v0 = k & ((1 << DD) - 1), v1 = (k + 1) & ((1 << DD) - 1);
        constexpr int e0 = ((k >> DD) << (DD + 1)) | v0, f0 = e0 | (1 << DD);
        constexpr int e1 = (((k + 1) >> DD) << (DD + 1)) | v1, f1 = e1 | (1 << DD);
        constexpr bool n0 = small_root_log<DD, v0, INV>() >= 96, n1 = small_root_log<DD, v1, INV>() >= 96;
        uint64_t a0 = n0 ? x[f0] : x[e0], b0 = n0 ? x[e0] : x[f0];
        uint64_t a1 = n1 ? x[f1] : x[e1], b1 = n1 ? x[e1] : x[f1];
        ar.add_sub2(a0, b0, a1, b1);
        ar.mul2(b0, w[v0], b1, w[v1]);
        x[e0] = a0;
        x[f0] = b0;
        x[e1] = a1;
        x[f1] = b1;
    });
}

// The twiddles of stages B0..B0 + K - 1 at the lane's place below register bit
// C + B0.
template <int M1, int B0, int K, bool INV>
__device__ __forceinline__ void first_twiddles(uint64_t (&b)[kTwoWords], const NttPass &a, uint32_t ch, uint32_t t)
{
    const uint32_t k = first_pos<M1>(a.s_lo, ch, t & ((1u << (kTwoTile - M1 + B0)) - 1));
#pragma unroll
    for (int dd = 0; dd < K; dd++) {
        const uint32_t lg = a.s_lo + B0 + dd + 1;
        b[dd] = gmem(cmem(a.tw_lg)[lg])[INV ? (0u - k) & ((1u << lg) - 1) : k];
    }
}

// Stages REM-1..0 of the first launch's M1; b: the twiddles of the round.
template <int M1, int REM, bool INV, class A>
__device__ __forceinline__ void first_rounds(A &ar, uint64_t *lds, uint64_t (&x)[1 << kTwoWords],
                                             const uint64_t (&b)[kTwoWords], const NttPass &a, uint32_t ch, uint32_t t)
{
    constexpr int LE = kTwoWords, C = kTwoTile - M1, E = 1 << LE;
    constexpr int K = REM > LE ? LE : REM, B0 = REM - K;
    constexpr int NEXT = B0 > LE ? B0 - LE : 0;
    uint64_t bn[LE];  // of the next round, in flight through this one
    if constexpr (B0 > 0) first_twiddles<M1, NEXT, B0 - NEXT, INV>(bn, a, ch, t);
    static_for<0, K>([&](auto kc) {
        constexpr int dd = K - 1 - decltype(kc)::value;
        root_stage<dd, INV, E>(ar, x, b[dd]);
    });
    if constexpr (B0 > 0) {
#pragma unroll
        for (int e = 0; e < E; e++) lds[lds_slot(column_pos<LE>(t, C + B0, e))] = x[e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < E; e++) x[e] = lds[lds_slot(column_pos<LE>(t, C + NEXT, e))];
        first_rounds<M1, B0, INV>(ar, lds, x, bn, a, ch, t);
    }
}

template <int M1, bool INV, class A>
__device__ __forceinline__ void first_transform(A &ar, uint64_t *lds, uint64_t (&x)[1 << kTwoWords], const NttPass &a,
                                                uint64_t tile, uint32_t t)
{
    constexpr int LE = kTwoWords, E = 1 << LE, C = kTwoTile - M1;
    const uint32_t s = a.s_lo, ch = (uint32_t)tile & ((1u << (s - C)) - 1);
    const uint64_t g = tile >> (s - C);  // block
    uint64_t b[LE];
    first_twiddles<M1, M1 - LE, LE, INV>(b, a, ch, t);
    auto pos = [&](int e) { return first_pos<M1>(s, ch, column_pos<LE>(t, kTwoTile - LE, e)); };
    uint64_t f[E];
    const gptr<const uint64_t> row = gmem(a.src) + ((a.mode == kSrcLde ? g >> a.rate : g) << a.L);
#pragma unroll
    for (int e = 0; e < E; e++) x[e] = A::load(row[pos(e)]);
    if (a.mode != kSrcInPlace) {
        const gptr<const uint64_t> fac =
            gmem(a.coset) + (a.mode == kSrcLde ? (g & ((1ull << a.rate) - 1)) << a.L : 0);
#pragma unroll
        for (int e = 0; e < E; e++) f[e] = fac[pos(e)];
#pragma unroll
        for (int e = 0; e < E; e += 2) ar.mul2(x[e], f[e], x[e + 1], f[e + 1]);
    }
    first_rounds<M1, M1, INV>(ar, lds, x, b, a, ch, t);
}

// src -> buf (the scratch), in the order of an in-place pass.
template <int M1, bool INV>
__global__ void __launch_bounds__(kTwoLanes) __attribute__((amdgpu_waves_per_eu(8)))
k_ntt_first(NttPass a)
{
    constexpr int LE = kTwoWords, C = kTwoTile - M1;
    __shared__ uint64_t lds[TwoShape::kSlots];
    const uint32_t t = threadIdx.x;
    const uint64_t tile = two_tile<C>(blockIdx.x);
    uint64_t x[1 << LE];
    Lazy lazy;
    first_transform<M1, INV>(lazy, lds, x, a, tile, t);
    const uint32_t s = a.s_lo, ch = (uint32_t)tile & ((1u << (s - C)) - 1);
    const gptr<uint64_t> row = gmem(a.buf) + ((tile >> (s - C)) << a.L);
#pragma unroll
    for (int e = 0; e < (1 << LE); e++) row[first_pos<M1>(s, ch, column_pos<LE>(t, C, e))] = x[e];
}

// The twiddles of stages B0..B0 + LE - 1 at the lane's place below bit B0.
template <int LE, int B0, bool INV>
__device__ __forceinline__ void second_twiddles(uint64_t (&b)[LE], const NttPass &a, uint32_t t)
{
    const uint32_t lo = t & ((1u << B0) - 1);
#pragma unroll
    for (int dd = 0; dd < LE; dd++) {
        b[dd] = gmem(cmem(a.tw_lg)[B0 + dd + 1])[INV ? (0u - lo) & ((1u << (B0 + dd + 1)) - 1) : lo];
    }
}

// Stages REM-1..0, the words of the first of these rounds in x and its
// twiddles in b; the last leaves the tile in x at register bit 0.
template <int LE, int REM, bool INV, class A>
__device__ __forceinline__ void second_rounds(A &ar, uint64_t *lds, uint64_t (&x)[1 << LE], const uint64_t (&b)[LE],
                                              const NttPass &a, uint32_t t)
{
    if constexpr (REM > LE) {
        constexpr int B0 = REM - LE, NEXT = B0 > LE ? B0 - LE : 0;
        uint64_t bn[LE];  // of the next round, in flight through this one
        if constexpr (B0 > LE) second_twiddles<LE, NEXT, INV>(bn, a, t);
        static_for<0, LE>([&](auto kc) {
            constexpr int dd = LE - 1 - decltype(kc)::value;
            root_stage<dd, INV, 1 << LE>(ar, x, b[dd]);
        });
#pragma unroll
        for (int e = 0; e < (1 << LE); e++) lds[lds_slot(column_pos<LE>(t, B0, e))] = x[e];
        __syncthreads();
#pragma unroll
        for (int e = 0; e < (1 << LE); e++) x[e] = lds[lds_slot(column_pos<LE>(t, NEXT, e))];
        second_rounds<LE, B0, INV>(ar, lds, x, bn, a, t);
    } else if constexpr (REM > 0) {
        last_stages<REM - 1, INV, 1 << LE>(ar, x);
    }
}

// Column and reversed row group of a second tile: it holds the rows
// x << (lg - 13) | g, and its output runs start at word gr << C of each
// 2^(lg - M2) words, gr the reversal of g.
template <int M2, bool INV, class A>
__device__ __forceinline__ void second_transform(A &ar, uint64_t *lds, const NttPass &a, const ColumnPost &post,
                                                 uint64_t tile, uint32_t t)
{
    constexpr int LE = kTwoWords, E = 1 << LE, C = kTwoTile - M2;
    const uint32_t gb = post.lg - kTwoTile, gr = (uint32_t)tile & ((1u << gb) - 1);
    const uint32_t g = __builtin_bitreverse32(gr) >> (32 - gb);
    const gptr<const uint64_t> col = gmem(a.src) + ((tile >> gb) << post.lg);
    uint64_t x[E], b[LE];
    second_twiddles<LE, M2 - LE, INV>(b, a, t);
#pragma unroll
    for (int e = 0; e < E; e++) {
        const uint32_t u = column_pos<LE>(t, M2 - LE, e);
        x[e] = A::load(col[((((u >> M2) << gb) | g) << M2) + (u & ((1u << M2) - 1))]);
    }
    second_rounds<LE, M2, INV>(ar, lds, x, b, a, t);
    // word u = t << LE | e goes to place rev(j) << C | rev(x) = rev(u) of the tile
    uint32_t to[E];
    const uint32_t r0 = __builtin_bitreverse32(t << LE);
#pragma unroll
    for (int e = 0; e < E; e++) to[e] = (r0 | __builtin_bitreverse32((uint32_t)e)) >> (32 - kTwoTile);
    if constexpr (INV) {
#pragma unroll
        for (int e = 0; e < E; e += 2) ar.mul2(x[e], post.scale, x[e + 1], post.scale);
        if (post.coset) {
            auto at = [&](int e) {
                return gmem(post.coset)[((to[e] >> C) << (post.lg - M2)) + (gr << C) + (to[e] & ((1u << C) - 1))];
            };
#pragma unroll
            for (int e = 0; e < E; e += 2) ar.mul2(x[e], at(e), x[e + 1], at(e + 1));
        }
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < E; e++) lds[lds_slot(to[e])] = A::result(x[e]);
}

// src (the scratch) -> buf, natural order.
template <int M2, bool INV>
__global__ void __launch_bounds__(kTwoLanes) __attribute__((amdgpu_waves_per_eu(8)))
k_ntt_second(NttPass a, ColumnPost post)
{
    constexpr int LE = kTwoWords, C = kTwoTile - M2;
    __shared__ uint64_t lds[TwoShape::kSlots];
    const uint32_t t = threadIdx.x;
    const uint64_t tile = two_tile<C>(blockIdx.x);
    Lazy lazy;
    second_transform<M2, INV>(lazy, lds, a, post, tile, t);
    __syncthreads();
    const uint32_t gb = post.lg - kTwoTile, gr = (uint32_t)tile & ((1u << gb) - 1);
    const gptr<uint64_t> col = gmem(a.buf) + ((tile >> gb) << post.lg) + (gr << C);
#pragma unroll
    for (int i = 0; i < (1 << LE); i++) {
        const uint32_t p = t + kTwoLanes * i;
        col[((p >> C) << (post.lg - M2)) + (p & ((1u << C) - 1))] = lds[lds_slot(p)];
    }
}

}  // namespace zkx
