// What the transform kernels share: their arithmetic on lazy values, the
// small-root stages, descriptors.
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
// Words are lazy (below 2^64) inside a transform and between its passes; a
// butterfly is 21 instructions and a test of two lane masks (gl64.h) rather
// than 30 on canonical words.  The last pass stores canonical ones.
//
// Bounds, 32 commits of 135 x 2^15 rate 3: the first pass, bound by its loads
// and stores (3.2 ms alone), 3.55 -> 3.53 ms; the 12-stage contiguous pass, of
// which they take 4.4, 5.93 -> 5.57.  (Redoing a whole tile exactly instead of
// fixing the lanes took 3.33 and 5.26 on random words, but 41 us against 27 for
// the inverse of 101 x 2^13 bits, as for any trace of small numbers.)
struct Lazy {
    static __device__ __forceinline__ uint64_t load(uint64_t x) { return x; }
    static __device__ __forceinline__ uint64_t result(uint64_t x) { return gl::canon(x); }
    __device__ __forceinline__ void add_sub2(uint64_t &x0, uint64_t &y0, uint64_t &x1, uint64_t &y1)
    {
        uint64_t s0, d0, s1, d1;
        gl::add_sub_lazy2(x0, y0, x1, y1, s0, d0, s1, d1);
        x0 = s0, y0 = d0, x1 = s1, y1 = d1;
    }
    __device__ __forceinline__ void mul2(uint64_t &x0, uint64_t w0, uint64_t &x1, uint64_t w1)
    {
        uint64_t r0, r1;
        gl::mul_fix2(x0, w0, x1, w1, r0, r1);
        x0 = r0, x1 = r1;
    }
    template <int E>
    __device__ __forceinline__ uint64_t shift(uint64_t x)
    {
        return gl::mul_pow2_lazy<E>(x);
    }
};

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
