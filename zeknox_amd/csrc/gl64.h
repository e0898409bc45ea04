// Goldilocks field p = 2^64 - 2^32 + 1 on the CDNA VALU.
//
// Values are u64 held in two VGPRs.  Every function takes and returns
// canonical values in [0, p) -- the representation the reference's digests
// and LDE outputs are compared in (ff/gl64_t.cuh:485-506 reduces to
// canonical; ff/goldilocks.hpp:139-177 keeps canonical values) -- unless its
// comment says otherwise.
//
// Instruction selection.  On gfx950 the 32-bit integer multiply-adds
// (v_mad_u64_u32, v_mul_hi_u32) issue at full rate, while the 64-bit VALU
// forms (v_lshl_add_u64, v_cmp_*_u64) run at about a third of it.  All
// additions and comparisons here are therefore written as 32-bit carry
// chains (__builtin_addc / __builtin_subc -> v_add_co_u32 / v_addc_co_u32,
// carries in SGPR masks, results picked with v_cndmask_b32), and products
// are built from four v_mad_u64_u32.  Reduction uses 2^64 = 2^32 - 1 and
// 2^96 = -1 (mod p).
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace gl {

constexpr uint64_t P = 0xFFFFFFFF00000001ull;
constexpr uint64_t EPS = 0xFFFFFFFFull;  // 2^64 mod p

__device__ __forceinline__ uint32_t lo32(uint64_t x) { return (uint32_t)x; }
__device__ __forceinline__ uint32_t hi32(uint64_t x) { return (uint32_t)(x >> 32); }
__device__ __forceinline__ uint64_t pack(uint32_t lo, uint32_t hi) { return ((uint64_t)hi << 32) | lo; }

// A wave-uniform constant the compiler cannot see through: it stays an SGPR
// operand of v_mad_u64_u32 instead of being strength-reduced into 64-bit
// shift-adds (which issue at about a third of the multiply-add rate).
__device__ __forceinline__ uint32_t opaque(uint32_t c)
{
    uint32_t r;
    asm("; opaque %0" : "=s"(r) : "0"(c));
    return r;
}

// A per-lane 64-bit value the compiler cannot see through (kept in a VGPR
// pair).  Placed after the first multiply-add of an accumulation chain it
// pins the chain's initial addend to that multiply-add, instead of letting
// the adds be reassociated into a trailing 64-bit add (v_lshl_add_u64, a
// third of the rate).
__device__ __forceinline__ uint64_t vopaque64(uint64_t x)
{
    asm("; vopaque %0" : "+v"(x));
    return x;
}

// x + y for y < 2^32 as one full-rate v_mad_u64_u32 (y * 1 + x); valid when
// the sum fits in 64 bits.
__device__ __forceinline__ uint64_t add_small(uint64_t x, uint32_t y) { return (uint64_t)y * opaque(1u) + x; }

// (a + b) mod p for a < 2^64 and b < p, canonical when either
//   a < p, or b <= 2^64 - 2^33 + 1 (then a may be any u64).
// s = a + b; t = s + EPS = s - p (mod 2^64); a + b >= p iff either carries.
__device__ __forceinline__ uint64_t add(uint64_t a, uint64_t b)
{
    uint32_t c1, c2, c3, c4;
    const uint32_t slo = __builtin_addc(lo32(a), lo32(b), 0u, &c1);
    const uint32_t shi = __builtin_addc(hi32(a), hi32(b), c1, &c2);
    const uint32_t tlo = __builtin_addc(slo, 0xFFFFFFFFu, 0u, &c3);
    const uint32_t thi = __builtin_addc(shi, 0u, c3, &c4);
    return (c2 | c4) ? pack(tlo, thi) : pack(slo, shi);
}

// (a - b) mod p for a, b < p: borrow -> add p, i.e. subtract EPS.
__device__ __forceinline__ uint64_t sub(uint64_t a, uint64_t b)
{
    uint32_t b1, b2, b3, b4;
    const uint32_t dlo = __builtin_subc(lo32(a), lo32(b), 0u, &b1);
    const uint32_t dhi = __builtin_subc(hi32(a), hi32(b), b1, &b2);
    const uint32_t tlo = __builtin_subc(dlo, 0xFFFFFFFFu, 0u, &b3);
    const uint32_t thi = __builtin_subc(dhi, 0u, b3, &b4);
    return b2 ? pack(tlo, thi) : pack(dlo, dhi);
}

// h * EPS = h * 2^32 - h for h < 2^32 (exact, <= 2^64 - 2^33 + 1).
__device__ __forceinline__ uint64_t mul_eps(uint32_t h)
{
    uint32_t b1, b2;
    const uint32_t ylo = __builtin_subc(0u, h, 0u, &b1);
    const uint32_t yhi = __builtin_subc(h, 0u, b1, &b2);
    return pack(ylo, yhi);
}

// Canonical residue of hi * 2^64 + lo (any 128-bit value):
//   hi * 2^64 = h0 * 2^64 + h1 * 2^96 = h0 * EPS - h1  (mod p).
__device__ __forceinline__ uint64_t reduce128(uint64_t lo, uint64_t hi)
{
    const uint32_t h0 = lo32(hi), h1 = hi32(hi);
    uint32_t b1, b2, b3, b4;
    const uint32_t xlo = __builtin_subc(lo32(lo), h1, 0u, &b1);
    const uint32_t xhi = __builtin_subc(hi32(lo), 0u, b1, &b2);
    // borrow: x = lo - h1 + 2^64, take off 2^64 = EPS (no underflow: x >= 2^64 - 2^32 + 1)
    const uint32_t elo = __builtin_subc(xlo, 0xFFFFFFFFu, 0u, &b3);
    const uint32_t ehi = __builtin_subc(xhi, 0u, b3, &b4);
    const uint64_t x = b2 ? pack(elo, ehi) : pack(xlo, xhi);
    return add(x, mul_eps(h0));
}

// Canonical residue of top * 2^64 + lo with top < 2^32.
__device__ __forceinline__ uint64_t reduce96(uint64_t lo, uint32_t top) { return add(lo, mul_eps(top)); }

// ---- carry-out forms
//
// v_mad_u64_u32 writes bit 64 of S0 * S1 + S2 to an SGPR lane mask; the
// compiler does not expose that carry, so the lazy reductions below reach it
// through inline asm.  gfx950 needs two wait states between a VALU write of
// a lane mask and a VALU read of it (the compiler inserts the same for its
// own carry chains): every mask is created and consumed inside one asm
// block, behind an s_nop 1, or leaves it two wait states after its write --
// except the product carry of mul128c, which is read by the second asm block
// of the reductions that take it: that block depends on
// the first one, whose inputs depend on the multiply-add writing the mask,
// so at least the first block's three instructions lie between them (a wait
// of its own would cost every product an issue slot; that the compiler does
// not spill it in between is checked in the machine code:
// tests/test_wait_states.py).  The
// inline constant -1 is 0xFFFFFFFF = EPS as the 32-bit multiplicand.

// Lazy residue (below 2^64, congruent mod p) of top * 2^64 + lo, top < 2^32:
// u = lo + top * EPS (mod 2^64, carry c: one v_mad_u64_u32), then
// u + c * EPS, which cannot carry again (c leaves u <= 2^64 - 2^33).
__device__ __forceinline__ uint64_t reduce96_lazy(uint64_t lo, uint32_t top)
{
    uint64_t u, r, s0, s1;
    uint32_t cv;
    asm("v_mad_u64_u32 %[u], %[s0], %[top], -1, %[lo]\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e64 %[cv], 0, 1, %[s0]\n\t"
        "v_mad_u64_u32 %[r], %[s1], %[cv], -1, %[u]"
        : [u] "=&v"(u), [r] "=&v"(r), [s0] "=&s"(s0), [s1] "=&s"(s1), [cv] "=&v"(cv)
        : [top] "v"(top), [lo] "v"(lo));
    return r;
}

// 64x64 -> 128 product from four multiply-adds, the carry of the middle sum
// left in a lane mask: a * b = lo + (hi + c * 2^32) * 2^64, c in {0, 1}
// (any a, b < 2^64).  u = a0 b0; v = a0 b1 + hi(u) (< 2^64); w = a1 b0 + v,
// whose bit 64 is c; hi = a1 b1 + hi(w) <= 2^64 - 2^32 (no carry).  Two
// instructions fewer than with the middle sum kept below 2^64 (a fifth
// multiply-add and a register-pair copy): the carry goes into the reduction as
// a borrow (reduce128c_lazy).
__device__ __forceinline__ void mul128c(uint64_t a, uint64_t b, uint64_t &lo, uint64_t &hi, uint64_t &c)
{
    const uint32_t a0 = lo32(a), a1 = hi32(a), b0 = lo32(b), b1 = hi32(b);
    const uint64_t u = (uint64_t)a0 * b0;
    const uint64_t v = (uint64_t)a0 * b1 + hi32(u);
    uint64_t w;
    asm("v_mad_u64_u32 %[w], %[c], %[x], %[y], %[v]"
        : [w] "=&v"(w), [c] "=&s"(c)
        : [x] "v"(a1), [y] "v"(b0), [v] "v"(v));
    hi = (uint64_t)a1 * b1 + hi32(w);
    lo = pack(lo32(u), lo32(w));
}

// A residue of hi * 2^64 + lo (any 128-bit value) below 2^64 but not
// necessarily below p ("lazy"):  hi * 2^64 = h0 * EPS - h1 (mod p).
//   u = lo + h0 * EPS (mod 2^64; carry c)      one v_mad_u64_u32
//   z = u - h1 (mod 2^64; borrow b)
//   r = z + (c - b) * EPS   -- each case lands in [0, 2^64): c without b
//       leaves z <= 2^64 - 2^33, b without c leaves z >= 2^64 - 2^32 + 1,
//       so the wrapped 64-bit sum is the exact value.  With cb = c - b in
//       {-1, 0, 1}: z + cb * EPS = (z - cb) + cb * 2^32, i.e. one signed
//       v_mad_i64_i32 (cb * -1 + z) and a 32-bit add to the high word.
__device__ __forceinline__ uint64_t reduce128_lazy(uint64_t lo, uint64_t hi)
{
    const uint32_t h0 = lo32(hi), h1 = hi32(hi);
    uint64_t u, sc;
    uint32_t cv;
    asm("v_mad_u64_u32 %[u], %[sc], %[h0], -1, %[lo]\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e64 %[cv], 0, 1, %[sc]"
        : [u] "=&v"(u), [sc] "=&s"(sc), [cv] "=&v"(cv)
        : [h0] "v"(h0), [lo] "v"(lo));
    uint32_t zlo, zhi, cb;
    uint64_t b1, b, bj;
    asm("v_sub_co_u32_e64 %[zlo], %[b1], %[ulo], %[h1]\n\t"
        "s_nop 1\n\t"
        "v_subb_co_u32_e64 %[zhi], %[b], %[uhi], 0, %[b1]\n\t"
        "s_nop 1\n\t"
        "v_subb_co_u32_e64 %[cb], %[bj], %[cv], 0, %[b]"
        : [zlo] "=&v"(zlo), [zhi] "=&v"(zhi), [cb] "=&v"(cb), [b1] "=&s"(b1), [b] "=&s"(b), [bj] "=&s"(bj)
        : [ulo] "v"(lo32(u)), [uhi] "v"(hi32(u)), [h1] "v"(h1), [cv] "v"(cv));
    uint64_t t, tj;
    asm("v_mad_i64_i32 %[t], %[tj], %[cb], -1, %[z]"
        : [t] "=&v"(t), [tj] "=&s"(tj)
        : [cb] "v"(cb), [z] "v"(pack(zlo, zhi)));
    // The high-word add stays in asm: written in C, the compiler folds it
    // into a following carry chain (canon's hi + 0 + carry becomes
    // hi(t) + cb + carry), whose carry-out then counts the wrap of this add.
    uint32_t rhi;
    asm("v_add_u32 %[r], %[a], %[b]" : [r] "=v"(rhi) : [a] "v"(hi32(t)), [b] "v"(cb));
    return pack(lo32(t), rhi);
}

// reduce128_lazy of lo + (hi + cin * 2^32) * 2^64 (cin a lane mask, the
// high word plus cin below 2^64): cin is the borrow into u - h1.
__device__ __forceinline__ uint64_t reduce128c_lazy(uint64_t lo, uint64_t hi, uint64_t cin)
{
    const uint32_t h0 = lo32(hi), h1 = hi32(hi);
    uint64_t u, sc;
    uint32_t cv;
    asm("v_mad_u64_u32 %[u], %[sc], %[h0], -1, %[lo]\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e64 %[cv], 0, 1, %[sc]"
        : [u] "=&v"(u), [sc] "=&s"(sc), [cv] "=&v"(cv)
        : [h0] "v"(h0), [lo] "v"(lo));
    uint32_t zlo, zhi, cb;
    uint64_t b1, b, bj;
    asm("v_subb_co_u32_e64 %[zlo], %[b1], %[ulo], %[h1], %[cin]\n\t"
        "s_nop 1\n\t"
        "v_subb_co_u32_e64 %[zhi], %[b], %[uhi], 0, %[b1]\n\t"
        "s_nop 1\n\t"
        "v_subb_co_u32_e64 %[cb], %[bj], %[cv], 0, %[b]"
        : [zlo] "=&v"(zlo), [zhi] "=&v"(zhi), [cb] "=&v"(cb), [b1] "=&s"(b1), [b] "=&s"(b), [bj] "=&s"(bj)
        : [ulo] "v"(lo32(u)), [uhi] "v"(hi32(u)), [h1] "v"(h1), [cv] "v"(cv), [cin] "s"(cin));
    uint64_t t, tj;
    asm("v_mad_i64_i32 %[t], %[tj], %[cb], -1, %[z]"
        : [t] "=&v"(t), [tj] "=&s"(tj)
        : [cb] "v"(cb), [z] "v"(pack(zlo, zhi)));
    // The high-word add stays in asm: written in C, the compiler folds it
    // into a following carry chain (canon's hi + 0 + carry becomes
    // hi(t) + cb + carry), whose carry-out then counts the wrap of this add.
    uint32_t rhi;
    asm("v_add_u32 %[r], %[a], %[b]" : [r] "=v"(rhi) : [a] "v"(hi32(t)), [b] "v"(cb));
    return pack(lo32(t), rhi);
}

// Two independent reduce128c_lazy at once: the same instructions with the two
// reductions interleaved, so every lane-mask read already sits two
// instructions after its write (one s_nop 0 per pair of steps instead of an
// s_nop 1 per step).
__device__ __forceinline__ void reduce128c_lazy2(uint64_t lo0, uint64_t hi0, uint64_t cin0, uint64_t lo1, uint64_t hi1,
                                                 uint64_t cin1, uint64_t &r0, uint64_t &r1)
{
    uint64_t u0, u1, sc0, sc1;
    uint32_t cv0, cv1;
    asm("v_mad_u64_u32 %[u0], %[sc0], %[a0], -1, %[l0]\n\t"
        "v_mad_u64_u32 %[u1], %[sc1], %[a1], -1, %[l1]\n\t"
        "s_nop 0\n\t"
        "v_cndmask_b32_e64 %[cv0], 0, 1, %[sc0]\n\t"
        "v_cndmask_b32_e64 %[cv1], 0, 1, %[sc1]"
        : [u0] "=&v"(u0), [u1] "=&v"(u1), [sc0] "=&s"(sc0), [sc1] "=&s"(sc1), [cv0] "=&v"(cv0), [cv1] "=&v"(cv1)
        : [a0] "v"(lo32(hi0)), [l0] "v"(lo0), [a1] "v"(lo32(hi1)), [l1] "v"(lo1));
    uint32_t zl0, zh0, cb0, zl1, zh1, cb1;
    uint64_t b10, b0, j0, b11, b1, j1;
    asm("v_subb_co_u32_e64 %[zl0], %[b10], %[ul0], %[h10], %[ci0]\n\t"
        "v_subb_co_u32_e64 %[zl1], %[b11], %[ul1], %[h11], %[ci1]\n\t"
        "s_nop 0\n\t"
        "v_subb_co_u32_e64 %[zh0], %[b0], %[uh0], 0, %[b10]\n\t"
        "v_subb_co_u32_e64 %[zh1], %[b1], %[uh1], 0, %[b11]\n\t"
        "s_nop 0\n\t"
        "v_subb_co_u32_e64 %[cb0], %[j0], %[cv0], 0, %[b0]\n\t"
        "v_subb_co_u32_e64 %[cb1], %[j1], %[cv1], 0, %[b1]"
        : [zl0] "=&v"(zl0), [zh0] "=&v"(zh0), [cb0] "=&v"(cb0), [zl1] "=&v"(zl1), [zh1] "=&v"(zh1),
          [cb1] "=&v"(cb1), [b10] "=&s"(b10), [b0] "=&s"(b0), [j0] "=&s"(j0), [b11] "=&s"(b11), [b1] "=&s"(b1),
          [j1] "=&s"(j1)
        : [ul0] "v"(lo32(u0)), [uh0] "v"(hi32(u0)), [h10] "v"(hi32(hi0)), [cv0] "v"(cv0), [ul1] "v"(lo32(u1)),
          [uh1] "v"(hi32(u1)), [h11] "v"(hi32(hi1)), [cv1] "v"(cv1), [ci0] "s"(cin0),
          [ci1] "s"(cin1));
    uint64_t t0, t1, tj0, tj1;
    asm("v_mad_i64_i32 %[t0], %[tj0], %[cb0], -1, %[z0]\n\t"
        "v_mad_i64_i32 %[t1], %[tj1], %[cb1], -1, %[z1]"
        : [t0] "=&v"(t0), [t1] "=&v"(t1), [tj0] "=&s"(tj0), [tj1] "=&s"(tj1)
        : [cb0] "v"(cb0), [z0] "v"(pack(zl0, zh0)), [cb1] "v"(cb1), [z1] "v"(pack(zl1, zh1)));
    uint32_t rh0, rh1;  // high-word adds kept in asm (see reduce128_lazy)
    asm("v_add_u32 %[r], %[a], %[b]" : [r] "=v"(rh0) : [a] "v"(hi32(t0)), [b] "v"(cb0));
    asm("v_add_u32 %[r], %[a], %[b]" : [r] "=v"(rh1) : [a] "v"(hi32(t1)), [b] "v"(cb1));
    r0 = pack(lo32(t0), rh0);
    r1 = pack(lo32(t1), rh1);
}

// x mod p for any x < 2^64 (x >= p iff x + EPS carries).
__device__ __forceinline__ uint64_t canon(uint64_t x)
{
    uint32_t c1, c2;
    const uint32_t tlo = __builtin_addc(lo32(x), 0xFFFFFFFFu, 0u, &c1);
    const uint32_t thi = __builtin_addc(hi32(x), 0u, c1, &c2);
    return c2 ? pack(tlo, thi) : x;
}

// a * b, lazy (below 2^64, congruent mod p) for any a, b < 2^64.
__device__ __forceinline__ uint64_t mul_lazy(uint64_t a, uint64_t b)
{
    uint64_t lo, hi, c;
    mul128c(a, b, lo, hi, c);
    return reduce128c_lazy(lo, hi, c);
}

// Two independent lazy products (their multiply-add chains and reductions
// interleave).
__device__ __forceinline__ void mul_lazy2(uint64_t a0, uint64_t b0, uint64_t a1, uint64_t b1, uint64_t &r0,
                                          uint64_t &r1)
{
    uint64_t lo0, hi0, c0, lo1, hi1, c1;
    mul128c(a0, b0, lo0, hi0, c0);
    mul128c(a1, b1, lo1, hi1, c1);
    reduce128c_lazy2(lo0, hi0, c0, lo1, hi1, c1, r0, r1);
}

// a * b, canonical (the lazy product's 7-instruction reduction plus the
// 4-instruction canonical fold is shorter than reduce128's chains).
__device__ __forceinline__ uint64_t mul(uint64_t a, uint64_t b) { return canon(mul_lazy(a, b)); }

// ---- multiplication by a power of two known at compile time
//
// 2 has order 192 mod p (2^96 = -1), and the 2^k-th roots of unity of the
// NTT for k <= 4 are powers of two (OMEGA[1..4] = 2^96, 2^48, 2^120, 2^156),
// so a butterfly whose twiddle is such a root multiplies by shifting.

constexpr uint64_t cmul(uint64_t a, uint64_t b) { return (uint64_t)((unsigned __int128)a * b % P); }
constexpr uint64_t cpow(uint64_t b, uint64_t e)
{
    uint64_t r = 1;
    for (; e; e >>= 1, b = cmul(b, b))
        if (e & 1) r = cmul(r, b);
    return r;
}
// OMEGA[k] = OMEGA[32]^(2^(32-k)) (gl64_params.hpp:48 gives OMEGA[32])
constexpr uint64_t kOmega32 = 1753635133440165772ull;
constexpr uint64_t comega(int k) { return cpow(kOmega32, 1ull << (32 - k)); }
// e with 2^e = w (mod p), -1 if w is not a power of two
constexpr int clog2(uint64_t w)
{
    for (int e = 0; e < 192; e++)
        if (cpow(2, e) == w) return e;
    return -1;
}

// x * 2^32, lazy: lo(x) * 2^32 + hi(x) * 2^64 = pack(0, lo(x)) + hi(x) * EPS.
__device__ __forceinline__ uint64_t shl32_lazy(uint64_t x) { return reduce96_lazy(pack(0u, lo32(x)), hi32(x)); }

// x^7 with the addition chain x2 = x^2, x3 = x*x2, x4 = x2^2, x7 = x3*x4;
// lazy in and out (any x < 2^64; result below 2^64, congruent mod p).  x3
// and x4 are independent products, computed as a pair.
__device__ __forceinline__ uint64_t pow7_lazy(uint64_t x)
{
    const uint64_t x2 = mul_lazy(x, x);
    uint64_t x3, x4;
    mul_lazy2(x2, x, x2, x2, x3, x4);
    return mul_lazy(x3, x4);
}

// x^7 and y^7 in lockstep (every product paired).
__device__ __forceinline__ void pow7_lazy2(uint64_t &x, uint64_t &y)
{
    uint64_t x2, y2, x3, y3, x4, y4;
    mul_lazy2(x, x, y, y, x2, y2);
    mul_lazy2(x2, x, y2, y, x3, y3);
    mul_lazy2(x2, x2, y2, y2, x4, y4);
    mul_lazy2(x3, x4, y3, y4, x, y);
}

// ---- products that leave a rare borrow to the caller
//
// In reduce128c_lazy the borrow b of u - h1 is all but impossible for a random
// product (u is below h1 < 2^32: 2^-32), yet folding it into the correction
// costs two of the seven instructions.  These forms leave it out,
//   r = z + c * EPS   (exact unless b),
// and or the borrow lanes into `bad`: a caller whose mask comes back nonzero
// throws the results away and takes the exact form.  The masks are or-ed
// where they are made, by the scalar unit, which waits for them: the compiler
// could take them through a VGPR, whose move needs wait states that it does
// not count after inline asm.  (A call with a mask that is not uniform does
// not compile.)  Per product 12
// instructions instead of 14; 32 commits of 135 x 2^15 51.4 -> 48.8 ms,
// Poseidon2 400 x 2^20 40.1 -> 38.0 ms (alternating builds).  A wave alone on
// its SIMD loses by it: it waits out the branches.

__device__ __forceinline__ uint64_t reduce128_rare(uint64_t lo, uint64_t hi, uint64_t cin, uint64_t &bad)
{
    uint64_t u, sc;
    uint32_t cv;
    asm("v_mad_u64_u32 %[u], %[sc], %[h0], -1, %[lo]\n\t"
        "s_nop 1\n\t"
        "v_cndmask_b32_e64 %[cv], 0, 1, %[sc]"
        : [u] "=&v"(u), [sc] "=&s"(sc), [cv] "=&v"(cv)
        : [h0] "v"(lo32(hi)), [lo] "v"(lo));
    uint32_t zlo, zhi;
    uint64_t b1, b;
    asm("v_subb_co_u32_e64 %[zlo], %[b1], %[ulo], %[h1], %[cin]\n\t"
        "s_nop 1\n\t"
        "v_subb_co_u32_e64 %[zhi], %[b], %[uhi], 0, %[b1]\n\t"
        "s_or_b64 %[bad], %[bad], %[b]"
        : [zlo] "=&v"(zlo), [zhi] "=&v"(zhi), [b1] "=&s"(b1), [b] "=&s"(b), [bad] "+s"(bad)
        : [ulo] "v"(lo32(u)), [uhi] "v"(hi32(u)), [h1] "v"(hi32(hi)), [cin] "s"(cin)
        : "scc");
    uint64_t r, j;
    asm("v_mad_u64_u32 %[r], %[j], %[cv], -1, %[z]" : [r] "=&v"(r), [j] "=&s"(j) : [cv] "v"(cv), [z] "v"(pack(zlo, zhi)));
    return r;
}

__device__ __forceinline__ void reduce128_rare2(uint64_t lo0, uint64_t hi0, uint64_t cin0, uint64_t lo1, uint64_t hi1,
                                                uint64_t cin1, uint64_t &r0, uint64_t &r1, uint64_t &bad, uint64_t &b0,
                                                uint64_t &b1)
{
    uint64_t u0, u1, sc0, sc1;
    uint32_t cv0, cv1;
    asm("v_mad_u64_u32 %[u0], %[sc0], %[a0], -1, %[l0]\n\t"
        "v_mad_u64_u32 %[u1], %[sc1], %[a1], -1, %[l1]\n\t"
        "s_nop 0\n\t"
        "v_cndmask_b32_e64 %[cv0], 0, 1, %[sc0]\n\t"
        "v_cndmask_b32_e64 %[cv1], 0, 1, %[sc1]"
        : [u0] "=&v"(u0), [u1] "=&v"(u1), [sc0] "=&s"(sc0), [sc1] "=&s"(sc1), [cv0] "=&v"(cv0), [cv1] "=&v"(cv1)
        : [a0] "v"(lo32(hi0)), [l0] "v"(lo0), [a1] "v"(lo32(hi1)), [l1] "v"(lo1));
    uint32_t zl0, zh0, zl1, zh1;
    uint64_t b10, b11;
    asm("v_subb_co_u32_e64 %[zl0], %[b10], %[ul0], %[h10], %[ci0]\n\t"
        "v_subb_co_u32_e64 %[zl1], %[b11], %[ul1], %[h11], %[ci1]\n\t"
        "s_nop 0\n\t"
        "v_subb_co_u32_e64 %[zh0], %[b0], %[uh0], 0, %[b10]\n\t"
        "v_subb_co_u32_e64 %[zh1], %[b1], %[uh1], 0, %[b11]\n\t"
        "s_or_b64 %[bad], %[bad], %[b0]\n\t"
        "s_or_b64 %[bad], %[bad], %[b1]"
        : [zl0] "=&v"(zl0), [zh0] "=&v"(zh0), [zl1] "=&v"(zl1), [zh1] "=&v"(zh1), [b10] "=&s"(b10), [b0] "=&s"(b0),
          [b11] "=&s"(b11), [b1] "=&s"(b1), [bad] "+s"(bad)
        : [ul0] "v"(lo32(u0)), [uh0] "v"(hi32(u0)), [h10] "v"(hi32(hi0)), [ul1] "v"(lo32(u1)), [uh1] "v"(hi32(u1)),
          [h11] "v"(hi32(hi1)), [ci0] "s"(cin0), [ci1] "s"(cin1)
        : "scc");
    uint64_t j0, j1;
    asm("v_mad_u64_u32 %[r], %[j], %[cv], -1, %[z]"
        : [r] "=&v"(r0), [j] "=&s"(j0)
        : [cv] "v"(cv0), [z] "v"(pack(zl0, zh0)));
    asm("v_mad_u64_u32 %[r], %[j], %[cv], -1, %[z]"
        : [r] "=&v"(r1), [j] "=&s"(j1)
        : [cv] "v"(cv1), [z] "v"(pack(zl1, zh1)));
}

__device__ __forceinline__ uint64_t mul_rare(uint64_t a, uint64_t b, uint64_t &bad)
{
    uint64_t lo, hi, c;
    mul128c(a, b, lo, hi, c);
    return reduce128_rare(lo, hi, c, bad);
}

__device__ __forceinline__ void mul_rare2(uint64_t a0, uint64_t b0, uint64_t a1, uint64_t b1, uint64_t &r0,
                                          uint64_t &r1, uint64_t &bad)
{
    uint64_t lo0, hi0, c0, lo1, hi1, c1, m0, m1;
    mul128c(a0, b0, lo0, hi0, c0);
    mul128c(a1, b1, lo1, hi1, c1);
    reduce128_rare2(lo0, hi0, c0, lo1, hi1, c1, r0, r1, bad, m0, m1);
}

// reduce96_lazy without its second step, which adds EPS in the lanes of
// `carry`: a carry out of lo + top * EPS needs lo above 2^64 - top * 2^32
// (for top < 2^16 one value in 2^16).  add_eps is that step.  The mask leaves
// the block, so its two wait states are in it: whatever the compiler reads it
// with next (the scalar unit, or a v_writelane_b32 that spills it) finds it.
__device__ __forceinline__ uint64_t reduce96_rare(uint64_t lo, uint32_t top, uint64_t &carry)
{
    uint64_t u;
    asm("v_mad_u64_u32 %[u], %[c], %[top], -1, %[lo]\n\t"
        "s_nop 1"
        : [u] "=&v"(u), [c] "=&s"(carry)
        : [top] "v"(top), [lo] "v"(lo));
    return u;
}
__device__ __forceinline__ uint64_t add_eps(uint64_t u, uint64_t lanes)
{
    uint64_t r, j;
    uint32_t cv;
    asm("s_nop 1\n\t"
        "v_cndmask_b32_e64 %[cv], 0, 1, %[m]\n\t"
        "v_mad_u64_u32 %[r], %[j], %[cv], -1, %[u]"
        : [r] "=&v"(r), [j] "=&s"(j), [cv] "=&v"(cv)
        : [u] "v"(u), [m] "s"(lanes));
    return r;
}

// ---- butterflies of transforms: sums, differences and products of lazy values
//
// A sum whose carry or a difference whose borrow has been folded in as EPS
// carries or borrows again only if an operand was not canonical, and a product
// borrows (reduce128_rare) once in 2^32 for random operands; but values of a
// trace are often small numbers, and small negative ones times the negative
// powers of two among the twiddles do it every time.  So the lanes are fixed in
// place behind a uniform branch, by one EPS: what was left out is added to (or
// taken from) the wrapped result, which is then exact.  A butterfly is 9
// instructions here and its product 12, against 12 and 18 in canonical form.

// x - EPS in the lanes of the mask.
__device__ __forceinline__ uint64_t sub_eps(uint64_t x, uint64_t lanes)
{
    uint32_t dlo, dhi, bv;
    uint64_t b;
    asm("s_nop 1\n\t"
        "v_cndmask_b32_e64 %[bv], 0, -1, %[m]\n\t"
        "v_sub_co_u32_e64 %[dlo], %[b], %[xl], %[bv]\n\t"
        "s_nop 1\n\t"
        "v_subb_co_u32_e64 %[dhi], %[b], %[xh], 0, %[b]"
        : [dlo] "=&v"(dlo), [dhi] "=&v"(dhi), [bv] "=&v"(bv), [b] "=&s"(b)
        : [xl] "v"(lo32(x)), [xh] "v"(hi32(x)), [m] "s"(lanes));
    return pack(dlo, dhi);
}

// s = a + b, d = a - b, for two pairs at once: every lane mask is read, or
// leaves its block, at least two instructions after its write.
__device__ __forceinline__ void add_sub_lazy2(uint64_t a0, uint64_t b0, uint64_t a1, uint64_t b1, uint64_t &s0,
                                              uint64_t &d0, uint64_t &s1, uint64_t &d1)
{
    uint32_t sl0, sh0, dl0, dh0, cv0, bv0, sl1, sh1, dl1, dh1, cv1, bv1;
    uint64_t mc0, mb0, mc1, mb1, any;
    asm("v_add_co_u32_e64 %[sl0], %[c0], %[al0], %[bl0]\n\t"
        "v_sub_co_u32_e64 %[dl0], %[b0], %[al0], %[bl0]\n\t"
        "v_add_co_u32_e64 %[sl1], %[c1], %[al1], %[bl1]\n\t"
        "v_sub_co_u32_e64 %[dl1], %[b1], %[al1], %[bl1]\n\t"
        "v_addc_co_u32_e64 %[sh0], %[c0], %[ah0], %[bh0], %[c0]\n\t"
        "v_subb_co_u32_e64 %[dh0], %[b0], %[ah0], %[bh0], %[b0]\n\t"
        "v_addc_co_u32_e64 %[sh1], %[c1], %[ah1], %[bh1], %[c1]\n\t"
        "v_subb_co_u32_e64 %[dh1], %[b1], %[ah1], %[bh1], %[b1]\n\t"
        "v_cndmask_b32_e64 %[cv0], 0, 1, %[c0]\n\t"
        "v_cndmask_b32_e64 %[bv0], 0, -1, %[b0]\n\t"
        "v_cndmask_b32_e64 %[cv1], 0, 1, %[c1]\n\t"
        "v_cndmask_b32_e64 %[bv1], 0, -1, %[b1]\n\t"
        "v_sub_co_u32_e64 %[dl0], %[b0], %[dl0], %[bv0]\n\t"
        "v_sub_co_u32_e64 %[dl1], %[b1], %[dl1], %[bv1]\n\t"
        "s_nop 0\n\t"
        "v_subb_co_u32_e64 %[dh0], %[b0], %[dh0], 0, %[b0]\n\t"
        "v_subb_co_u32_e64 %[dh1], %[b1], %[dh1], 0, %[b1]\n\t"
        "s_or_b64 %[any], %[b0], %[b1]\n\t"
        "s_nop 0"
        : [sl0] "=&v"(sl0), [sh0] "=&v"(sh0), [dl0] "=&v"(dl0), [dh0] "=&v"(dh0), [cv0] "=&v"(cv0), [bv0] "=&v"(bv0),
          [sl1] "=&v"(sl1), [sh1] "=&v"(sh1), [dl1] "=&v"(dl1), [dh1] "=&v"(dh1), [cv1] "=&v"(cv1), [bv1] "=&v"(bv1),
          [c0] "=&s"(mc0), [b0] "=&s"(mb0), [c1] "=&s"(mc1), [b1] "=&s"(mb1), [any] "=&s"(any)
        : [al0] "v"(lo32(a0)), [ah0] "v"(hi32(a0)), [bl0] "v"(lo32(b0)), [bh0] "v"(hi32(b0)), [al1] "v"(lo32(a1)),
          [ah1] "v"(hi32(a1)), [bl1] "v"(lo32(b1)), [bh1] "v"(hi32(b1))
        : "scc");
    uint64_t k0, k1;
    asm("v_mad_u64_u32 %[r0], %[k0], %[cv0], -1, %[s0]\n\t"
        "v_mad_u64_u32 %[r1], %[k1], %[cv1], -1, %[s1]\n\t"
        "s_or_b64 %[any], %[any], %[k0]\n\t"
        "s_or_b64 %[any], %[any], %[k1]"
        : [r0] "=&v"(s0), [k0] "=&s"(k0), [r1] "=&v"(s1), [k1] "=&s"(k1), [any] "+s"(any)
        : [cv0] "v"(cv0), [s0] "v"(pack(sl0, sh0)), [cv1] "v"(cv1), [s1] "v"(pack(sl1, sh1))
        : "scc");
    d0 = pack(dl0, dh0);
    d1 = pack(dl1, dh1);
    if (__builtin_expect(any != 0, 0)) {
        s0 = add_eps(s0, k0);
        s1 = add_eps(s1, k1);
        d0 = sub_eps(d0, mb0);
        d1 = sub_eps(d1, mb1);
    }
}

// Two products, exact (lazy).
__device__ __forceinline__ void mul_fix2(uint64_t a0, uint64_t w0, uint64_t a1, uint64_t w1, uint64_t &r0, uint64_t &r1)
{
    uint64_t lo0, hi0, c0, lo1, hi1, c1, b0, b1, any = 0;
    mul128c(a0, w0, lo0, hi0, c0);
    mul128c(a1, w1, lo1, hi1, c1);
    reduce128_rare2(lo0, hi0, c0, lo1, hi1, c1, r0, r1, any, b0, b1);
    if (__builtin_expect(any != 0, 0)) {
        r0 = sub_eps(r0, b0);
        r1 = sub_eps(r1, b1);
    }
}

// x * 2^E, lazy, for E < 96 and any x < 2^64: with x * 2^(E mod 32) =
// x0 + x1 * 2^32 + x2 * 2^64 (x2 < 2^32),
//   E < 32       x0 + x1 * 2^32 + x2 * EPS
//   32 <= E < 64 x0 * 2^32 + x1 * EPS - x2
//   64 <= E      x0 * EPS - (x1 + x2 * 2^32).
template <int E>
__device__ __forceinline__ uint64_t mul_pow2_lazy(uint64_t x)
{
    static_assert(E >= 0 && E < 96, "exponent below half the order of 2");
    constexpr int s = E % 32;
    const uint64_t l = x << s;
    const uint32_t x2 = s ? (uint32_t)(x >> ((64 - s) & 63)) : 0u;
    if constexpr (E == 0) return x;
    else if constexpr (E < 32) return reduce96_lazy(l, x2);
    else if constexpr (E == 32) return shl32_lazy(x);
    else if constexpr (E < 64) {
        // lo + hi * 2^64 with lo = x0 * 2^32, hi = (x1, x2)
        return reduce128_lazy(pack(0u, lo32(l)), pack(hi32(l), x2));
    } else {
        // the subtrahend is below 2^62, so the second borrow cannot be: a
        // first one leaves at least 2^64 - 2^62
        static_assert(s <= 30, "x2 below 2^30");
        const uint64_t y = mul_eps(lo32(l));
        uint32_t dlo, dhi, bv;
        uint64_t b;
        asm("v_sub_co_u32_e64 %[dlo], %[b], %[yl], %[h0]\n\t"
            "s_nop 1\n\t"
            "v_subb_co_u32_e64 %[dhi], %[b], %[yh], %[h1], %[b]\n\t"
            "s_nop 1\n\t"
            "v_cndmask_b32_e64 %[bv], 0, -1, %[b]\n\t"
            "v_sub_co_u32_e64 %[dlo], %[b], %[dlo], %[bv]\n\t"
            "s_nop 1\n\t"
            "v_subb_co_u32_e64 %[dhi], %[b], %[dhi], 0, %[b]"
            : [dlo] "=&v"(dlo), [dhi] "=&v"(dhi), [bv] "=&v"(bv), [b] "=&s"(b)
            : [yl] "v"(lo32(y)), [yh] "v"(hi32(y)), [h0] "v"(hi32(l)), [h1] "v"(x2));
        return pack(dlo, dhi);
    }
}

// x^7 of a wave whose branch is uniform: the products above, and the exact
// ones for the whole wave if any lane borrowed.  `carry`: lanes in which x
// still lacks an EPS (reduce96_rare).
__device__ __forceinline__ uint64_t pow7_wave(uint64_t x, uint64_t carry = 0)
{
    uint64_t bad = carry, x3, x4;
    const uint64_t x2 = mul_rare(x, x, bad);
    mul_rare2(x2, x, x2, x2, x3, x4, bad);
    uint64_t r = mul_rare(x3, x4, bad);
    if (__builtin_expect(bad != 0, 0)) r = pow7_lazy(add_eps(x, carry));
    return r;
}

// x^7 and y^7 in lockstep.
__device__ __forceinline__ void pow7_wave2(uint64_t &x, uint64_t &y)
{
    uint64_t bad = 0, x2, y2, x3, y3, x4, y4, xr, yr;
    mul_rare2(x, x, y, y, x2, y2, bad);
    mul_rare2(x2, x, y2, y, x3, y3, bad);
    mul_rare2(x2, x2, y2, y2, x4, y4, bad);
    mul_rare2(x3, x4, y3, y4, xr, yr, bad);
    if (__builtin_expect(bad != 0, 0)) {
        pow7_lazy2(x, y);
    } else {
        x = xr;
        y = yr;
    }
}

// x^7, canonical.
__device__ __forceinline__ uint64_t pow7(uint64_t x)
{
    const uint64_t x2 = mul(x, x);
    const uint64_t x3 = mul(x2, x);
    const uint64_t x4 = mul(x2, x2);
    return mul(x3, x4);
}

__device__ __forceinline__ uint64_t pow(uint64_t b, uint64_t e)
{
    uint64_t r = 1;
    while (e) {
        if (e & 1) r = mul(r, b);
        b = mul(b, b);
        e >>= 1;
    }
    return r;
}

}  // namespace gl
