// What the transform kernels share: their arithmetic on lazy values, the
// second computation of a tile, the small-root stages, descriptors.
#pragma once
#include <type_traits>

#include "gl64.h"
#include "gmem.h"
#include "ntt_types.h"

namespace zkx {

// LDS slot of tile position u (one pad word per 32 breaks power-of-two strides)
__device__ __forceinline__ uint32_t lds_slot(uint32_t u) { return u + (u >> 5); }

// ---- arithmetic of the passes
//
// A butterfly is 21 instructions on lazy values (Lazy) rather than 30 on
// canonical ones (Exact): what a random operand needs once in 2^32 is left
// out and its lanes noted in `bad` (gl64.h).  A tile with such a lane is
// computed again with Exact, from the source that nothing has overwritten
// yet.  Words between the passes of a transform are lazy too; the contiguous
// pass, the last, stores canonical ones.
//
// Bounds, 64 x 2^20 forward (1.07 GB of traffic a pass): the 12-stage
// contiguous pass 375 -> 318 us, of which its loads and stores alone take
// 273; the 8-stage strided pass 298 -> 294 us, bound by its loads and stores
// (250 alone).  The whole transform 906 -> 854 us, alternating builds.

struct Lazy {
    uint64_t bad;
    // (zero from the scalar unit: as a constant it may join the masks of
    // another branch in a VGPR)
    __device__ __forceinline__ Lazy() { asm("s_mov_b64 %0, 0" : "=s"(bad)); }
    static __device__ __forceinline__ uint64_t load(uint64_t x) { return x; }
    static __device__ __forceinline__ uint64_t result(uint64_t x) { return gl::canon(x); }
    __device__ __forceinline__ void add_sub2(uint64_t &x0, uint64_t &y0, uint64_t &x1, uint64_t &y1)
    {
        uint64_t s0, d0, s1, d1;
        gl::add_sub_rare2(x0, y0, x1, y1, s0, d0, s1, d1, bad);
        x0 = s0, y0 = d0, x1 = s1, y1 = d1;
    }
    __device__ __forceinline__ void mul2(uint64_t &x0, uint64_t w0, uint64_t &x1, uint64_t w1)
    {
        uint64_t r0, r1;
        gl::mul_rare2(x0, w0, x1, w1, r0, r1, bad);
        x0 = r0, x1 = r1;
    }
    __device__ __forceinline__ uint64_t mul(uint64_t x, uint64_t w) { return gl::mul_rare(x, w, bad); }
    template <int E>
    __device__ __forceinline__ uint64_t shift(uint64_t x)
    {
        return gl::mul_pow2_rare<E>(x, bad);
    }
};

struct Exact {
    static __device__ __forceinline__ uint64_t load(uint64_t x) { return gl::canon(x); }
    static __device__ __forceinline__ uint64_t result(uint64_t x) { return x; }
    __device__ __forceinline__ void add_sub2(uint64_t &x0, uint64_t &y0, uint64_t &x1, uint64_t &y1)
    {
        const uint64_t s0 = gl::add(x0, y0), d0 = gl::sub(x0, y0), s1 = gl::add(x1, y1), d1 = gl::sub(x1, y1);
        x0 = s0, y0 = d0, x1 = s1, y1 = d1;
    }
    __device__ __forceinline__ void mul2(uint64_t &x0, uint64_t w0, uint64_t &x1, uint64_t w1)
    {
        x0 = mul(x0, w0);
        x1 = mul(x1, w1);
    }
    // (the form with the fewest live registers)
    __device__ __forceinline__ uint64_t mul(uint64_t x, uint64_t w) { return gl::mul_nc(x, w); }
    template <int E>
    __device__ __forceinline__ uint64_t shift(uint64_t x)
    {
        // (x is canonical; the compiler folds a canon() that directly follows a
        // sub() into its carry chain and counts the wrap of that as its own)
        if constexpr (E == 0) return x;
        else return gl::mul_pow2<E>(x);
    }
};

// The lane and tile of the second computation, through values the compiler
// cannot see through: nothing the first one loaded or computed stays in
// registers for it.
__device__ __forceinline__ void again(uint32_t &t, uint64_t &tile)
{
    asm volatile("; again %0 %1" : "+v"(t), "+s"(tile));
}

// Whether any wave of the work-group noted a lane; ends with every LDS write
// before it visible.
template <int LANES = kNttThreads>
__device__ __forceinline__ bool barrier_any(uint32_t *flags, uint64_t bad)
{
    if ((threadIdx.x & 63) == 0) flags[threadIdx.x >> 6] = bad != 0 ? 1u : 0u;
    __syncthreads();
    uint32_t any = 0;
#pragma unroll
    for (int i = 0; i < LANES / 64; i++) any |= flags[i];
    return __builtin_amdgcn_readfirstlane(any) != 0;
}

// ---- stages whose twiddles are roots of order <= 16: w = 1 (no product) or
// a power of two (a shift; 2^96 = -1 is the difference taken the other way
// round)

template <int I, int N, class F>
__device__ __forceinline__ void static_for(F &&f)
{
    if constexpr (I < N) {
        f(std::integral_constant<int, I>{});
        static_for<I + 1, N>(f);
    }
}

// e with 2^e = w_{2^(D+1)}^V (w^-V for the inverse)
template <int D, int V, bool INV>
constexpr int small_root_log()
{
    constexpr int L = gl::clog2(gl::comega(D + 1));
    static_assert(L >= 0, "the 2^(D+1)-th root of unity of the transform is a power of two");
    constexpr int E0 = (V * L) % 192;
    return INV ? (192 - E0) % 192 : E0;
}

template <int DD, bool INV, int E, class A>
__device__ __forceinline__ void last_stages(A &ar, uint64_t (&x)[E])
{
    static_for<0, E / 4>([&](auto kc) {
        constexpr int k = 2 * decltype(kc)::value;
        constexpr int e0 = ((k >> DD) << (DD + 1)) | (k & ((1 << DD) - 1)), f0 = e0 | (1 << DD);
        constexpr int e1 = (((k + 1) >> DD) << (DD + 1)) | ((k + 1) & ((1 << DD) - 1)), f1 = e1 | (1 << DD);
        constexpr int E0 = small_root_log<DD, (e0 & ((1 << DD) - 1)), INV>();
        constexpr int E1 = small_root_log<DD, (e1 & ((1 << DD) - 1)), INV>();
        uint64_t a0 = E0 >= 96 ? x[f0] : x[e0], b0 = E0 >= 96 ? x[e0] : x[f0];
        uint64_t a1 = E1 >= 96 ? x[f1] : x[e1], b1 = E1 >= 96 ? x[e1] : x[f1];
        ar.add_sub2(a0, b0, a1, b1);
        x[e0] = a0;
        x[e1] = a1;
        x[f0] = ar.template shift<E0 % 96>(b0);
        x[f1] = ar.template shift<E1 % 96>(b1);
    });
    if constexpr (DD > 0) last_stages<DD - 1, INV, E>(ar, x);
}

// ---- descriptors
//
// A launch's descriptor list is read through the constant address space
// (scalar loads into SGPRs; as vector loads they cost 32 VGPRs).

__device__ __forceinline__ NttPass pass_at(const NttPass *passes, uint32_t npasses, const NttPass &one, uint64_t b)
{
    if (!npasses) return one;
    const cptr<NttPass> cp = cmem(passes);
    uint32_t lo = 0, hi = npasses;
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (cp[mid].tile_begin <= b) lo = mid;
        else hi = mid;
    }
    static_assert(sizeof(NttPass) % 8 == 0, "descriptor copied as 64-bit words");
    constexpr int W = sizeof(NttPass) / 8;
    const cptr<uint64_t> src = (cptr<uint64_t>)(cp + lo);
    uint64_t w[W];
#pragma unroll
    for (int i = 0; i < W; i++) w[i] = src[i];
    NttPass r;
    __builtin_memcpy(&r, w, sizeof r);
    return r;
}

}  // namespace zkx
