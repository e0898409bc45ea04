// Poseidon and Poseidon2 (Goldilocks, width 12; poseidon/poseidon.cu:563-838,
// poseidon2/poseidon2.cu:65-209) with every linear map on the matrix cores,
// 64 permutations per wave.
//
// The maps between S-boxes (mfma_tables.h) are exact integer products of
// bytes: the state's 64-bit slots are cut into their 8 bytes, a coefficient
// and a byte give eight signed digits, and v_mfma_i32_32x32x32_i8 sums them.
// The vector unit recombines eight digit sums per output element.
//
// Wave layout.  A wave holds two groups t of 32 permutations, two lanes per
// permutation: lane l (column j = l & 31, half h = l >> 5) holds elements
// 6h..6h + 5 of permutation (t, j).  v_mfma_i32_32x32x32_i8 (gfx950, layout
// measured) computes D[i][j] = sum_{h, q} A_{32h+i}[q] * B_{32h+j}[q] over
// the 16 bytes q each lane supplies, and lane 32h' + j receives D[i][j] for
// i = 8k + 4h' + r in its register 4k + r.  So a lane supplies its own slots
// as B, and with the rows ordered by M-block as in mfma_tables.h it receives
// the eight digit sums of its own elements 2 beta, 2 beta + 1.
//
// Partial rounds.  A group of five: the sums of x_2..x_5 come first (one
// M-block: x_2, x_3 on half 0 and x_4, x_5 on half 1, for both groups), and
// v_permlane32_swap hands each lane those of one permutation, (h, j): every
// lane then runs one permutation's five S-boxes, adding the earlier outputs
// of the group itself (h_{j-i} y_i), swaps the outputs back into their slots
// and the group's map gives the next state.  One recombination of twelve
// elements per five rounds instead of one per round: 12 layers of vector
// work instead of 30.
//
// Bound: VALU issue (1.03 of one wave instruction per 4 cycles per SIMD, the
// MFMAs beside it; multiply-adds, carries and three-operand forms take 4
// cycles, moves and plain adds 2).  Against one layer per round (the MDS on the matrix
// cores for Poseidon, everything on the VALU for Poseidon2), wave
// instructions per leaf permutation: Poseidon 205 -> 153 VALU, 8.4 -> 4.3
// MFMA; Poseidon2 234 -> 162 VALU.  Leaf launch of 32 x 2^18 leaves of 135:
// 56.4 -> 41.0 ms; of 2^21 leaves of 400 with Poseidon2: 36 -> 31.7 ms.
// The S-boxes' products and the recombination then leave their rare corrections
// to a branch (gl64.h): 153 -> 137 VALU and 41.0 -> 38.6 ms, Poseidon2 162 ->
// 146 and 31.7 -> 29.7 ms.  With a chunk's loads together (merkle_kernels.h) 133
// VALU and 36.8 ms, Poseidon2 28.5 ms.
// Five rounds: the map of four leaves a K-chunk unused and costs as much; six
// needs a fifth chunk and weights beyond 32 bits.
//
// Recombination (per output element, lazy in and out, as hash.h):
//   L = KL + (D0 + 2^8 D1) + 2^16 (D2 + 2^8 D3),  H = KH + (same on D4..D7),
// with KL, KH the map's constant pair (which keeps both non-negative), then
// limb_combine(L, H) (0 <= L, H < 2^47).  The chains run in signed 32x32+64
// multiply-adds.
//
// (Accumulator chains stay within one opcode, in place.  Observed: a 16x16x64
// result taken as the accumulator of a 16x16x32 product, issued with no wait
// states between them, came out wrong; why is not established, and no kernel
// does it.)
#pragma once
#include "hash.h"
#include "mfma_tables.h"

namespace zkx {

typedef int mf_v4i __attribute__((ext_vector_type(4)));
typedef int mf_v16i __attribute__((ext_vector_type(16)));

// The tables in device memory; kernels that do not hash with HT never name
// them, so each translation unit holds its own hash's alone.
template <int HT>
__device__ const mfma::Tables c_mfma = mfma::make<HT>();

// What a work-group keeps of them in LDS: the operands used all the time
// (24 KiB) and the constant rows.
struct MfmaLds {
    mf_v4i op[mfma::kOpsLds][64];
    alignas(16) uint64_t row[mfma::kRows][12][2];
};

// dst <- src, COUNT 16-byte words by a work-group of N lanes: every load in
// flight before the first write.
template <int COUNT, int N>
__device__ __forceinline__ void copy_to_lds(mf_v4i *dst, const mf_v4i *src)
{
    constexpr int kSteps = (COUNT + N - 1) / N;
    const uint32_t t = threadIdx.x;
    mf_v4i v[kSteps];
#pragma unroll
    for (int i = 0; i < kSteps; i++)
        if (COUNT % N == 0 || t + i * N < COUNT) v[i] = src[t + i * N];
#pragma unroll
    for (int i = 0; i < kSteps; i++)
        if (COUNT % N == 0 || t + i * N < COUNT) dst[t + i * N] = v[i];
}

template <int HT, int N>
__device__ __forceinline__ void mfma_fill(MfmaLds &m)
{
    copy_to_lds<mfma::kOpsLds * 64, N>(&m.op[0][0], reinterpret_cast<const mf_v4i *>(c_mfma<HT>.op));
    copy_to_lds<mfma::kRows * 12, N>(reinterpret_cast<mf_v4i *>(m.row), reinterpret_cast<const mf_v4i *>(c_mfma<HT>.row));
}

// Exchanges the upper half of a with the lower half of b: a becomes
// (a of half 0, b of half 0), b becomes (a of half 1, b of half 1).
// v_permlane32_swap_b32 needs two wait states after a VALU write of its
// operands; the compiler does not count the writes of inline asm (the
// reductions of gl64.h end in one), so the wait is part of the block.
__device__ __forceinline__ void swap_halves(uint64_t &a, uint64_t &b)
{
    uint32_t a0 = gl::lo32(a), a1 = gl::hi32(a), b0 = gl::lo32(b), b1 = gl::hi32(b);
    asm("s_nop 1\n\t"
        "v_permlane32_swap_b32 %[a0], %[b0]\n\t"
        "v_permlane32_swap_b32 %[a1], %[b1]"
        : [a0] "+v"(a0), [a1] "+v"(a1), [b0] "+v"(b0), [b1] "+v"(b1));
    a = gl::pack(a0, a1);
    b = gl::pack(b0, b1);
}
__device__ __forceinline__ void swap_halves(uint32_t (&a)[4], uint32_t (&b)[4])
{
    asm("s_nop 1\n\t"
        "v_permlane32_swap_b32 %[a0], %[b0]\n\t"
        "v_permlane32_swap_b32 %[a1], %[b1]\n\t"
        "v_permlane32_swap_b32 %[a2], %[b2]\n\t"
        "v_permlane32_swap_b32 %[a3], %[b3]"
        : [a0] "+v"(a[0]), [a1] "+v"(a[1]), [a2] "+v"(a[2]), [a3] "+v"(a[3]), [b0] "+v"(b[0]), [b1] "+v"(b[1]),
          [b2] "+v"(b[2]), [b3] "+v"(b[3]));
}

// A slot's bytes as the MFMA takes them (u - 128, signed).
__device__ __forceinline__ uint64_t mfma_bytes(uint64_t x) { return x ^ 0x8080808080808080ull; }

__device__ __forceinline__ mf_v4i mfma_pair(uint64_t x0, uint64_t x1)
{
    return mf_v4i{(int)gl::lo32(x0), (int)gl::hi32(x0), (int)gl::lo32(x1), (int)gl::hi32(x1)};
}

// D0 + 2^8 D1 of two digit sums.
__device__ __forceinline__ uint32_t digit_pair(int d0, int d1) { return (uint32_t)d0 + ((uint32_t)d1 << 8); }

// Keeps the operands of an MFMA chain in their registers until p, computed
// from the chain's result, is there.  Observed: without it, where the compiler
// put a v_mov over a register of a chain's A operand right after the MFMA that
// reads it, the sums came out wrong with two or more waves on the SIMD (in the
// second group of a wave), and right with it.  The cause is not established:
// the documented waits after an MFMA cover its accumulator, not A and B, and
// the compiler counts none for them.  Every chain holds its operands, so no
// kernel depends on the answer.
template <int NK>
__device__ __forceinline__ void hold_operands(const mf_v4i (&a)[NK], const mf_v4i (&b)[NK], uint32_t p)
{
#pragma unroll
    for (int kappa = 0; kappa < NK; kappa++) asm volatile("; hold %0 %1 %2" ::"v"(p), "v"(a[kappa]), "v"(b[kappa]));
}

// limb_combine (any A and B with B + hi(A) below 2^64; the sums here are below
// 2^63), less the EPS of the lanes of `carry`, which are the rarer the smaller
// B is: about one value in 2^64 / B.
__device__ __forceinline__ uint64_t limb_combine_rare(uint64_t A, uint64_t B, uint64_t &carry)
{
    const uint64_t T = gl::add_small(B, gl::hi32(A));
    return gl::reduce96_rare(gl::pack(gl::lo32(A), gl::lo32(T)), gl::hi32(T), carry);
}

// p01 + 2^16 p23 + k, in signed multiply-adds.
__device__ __forceinline__ uint64_t half_sum(uint32_t p01, uint32_t p23, uint64_t k)
{
    const int64_t one = (int32_t)gl::opaque(1u), m16 = (int32_t)gl::opaque(65536u);
    const uint64_t s = gl::vopaque64((uint64_t)((int64_t)(int32_t)p01 * one + (int64_t)k));
    return gl::vopaque64((uint64_t)((int64_t)(int32_t)p23 * m16 + (int64_t)s));
}

// s <- the map with operands `op` (this lane's, [M-block][K-chunk] 64 lanes
// apart) on the slots b, plus the constants `row` of this lane's elements.
template <int NK>
__device__ __forceinline__ void mfma_map(uint64_t s[2][6], const mf_v4i (&b)[2][NK], const mf_v4i *op,
                                         const uint64_t (*row)[2])
{
    // one M-block and group at a time, recombined as soon as its chain is
    // done: 16 accumulator VGPRs live
    uint64_t carry[2][6];
#pragma unroll
    for (int beta = 0; beta < 3; beta++) {
        mf_v4i a[NK];
#pragma unroll
        for (int kappa = 0; kappa < NK; kappa++) a[kappa] = op[(beta * NK + kappa) * 64];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            mf_v16i dd = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[0], b[t][0], mf_v16i{}, 0, 0, 0);
#pragma unroll
            for (int kappa = 1; kappa < NK; kappa++)
                dd = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[kappa], b[t][kappa], dd, 0, 0, 0);
            hold_operands<NK>(a, b[t], digit_pair(dd[0], dd[1]));
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const int e = 2 * beta + u, q = 8 * u;
                const uint64_t L = half_sum(digit_pair(dd[q], dd[q + 1]), digit_pair(dd[q + 2], dd[q + 3]), row[e][0]);
                const uint64_t H =
                    half_sum(digit_pair(dd[q + 4], dd[q + 5]), digit_pair(dd[q + 6], dd[q + 7]), row[e][1]);
                s[t][e] = limb_combine_rare(L, H, carry[t][e]);
            }
        }
    }
    uint64_t any = 0;
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int e = 0; e < 6; e++) any |= carry[t][e];
    if (__builtin_expect(any != 0, 0)) {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int e = 0; e < 6; e++) s[t][e] = gl::add_eps(s[t][e], carry[t][e]);
    }
}

// The digit pairs of the outputs of one M-block: x[t][u] for this lane's
// half, swapped so that x[h'][u] is output 2h' + u of permutation (h, j).
__device__ __forceinline__ void mfma_outputs(uint32_t (&x)[2][2][4], const mf_v4i (&b)[2][3], const mf_v4i *op)
{
    mf_v4i a[3];
#pragma unroll
    for (int kappa = 0; kappa < 3; kappa++) a[kappa] = op[kappa * 64];
#pragma unroll
    for (int t = 0; t < 2; t++) {
        mf_v16i dd = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[0], b[t][0], mf_v16i{}, 0, 0, 0);
        dd = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[1], b[t][1], dd, 0, 0, 0);
        dd = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[2], b[t][2], dd, 0, 0, 0);
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int n = 0; n < 4; n++) x[t][u][n] = digit_pair(dd[8 * u + 2 * n], dd[8 * u + 2 * n + 1]);
        hold_operands<3>(a, b[t], x[t][0][0]);
    }
#pragma unroll
    for (int u = 0; u < 2; u++) swap_halves(x[0][u], x[1][u]);
}

// An S-box input: the recombined output (digit pairs d, constant k) plus
// sum_i h[m - i] y[i] over the m earlier outputs of its group.  Weights below
// 2^32 enter the recombination as multiply-adds of the output's halves (their
// sum is below 2^30); larger ones as lazy products.
template <int HT>
constexpr uint64_t mfma_h(int m)
{
    constexpr auto h = mfma::partial_weights<HT>();
    return h.v[m];
}

// The sum of the weights up to h_last (2^32 if one of them is larger).
template <int HT>
constexpr uint64_t mfma_h_sum(int last)
{
    uint64_t s = 0;
    for (int m = 1; m <= last; m++) s += mfma_h<HT>(m) < (1ull << 32) ? mfma_h<HT>(m) : 1ull << 32;
    return s < (1ull << 32) ? s : 1ull << 32;
}
static_assert(mfma_h_sum<kPoseidon>(mfma::kGroupRounds - 1) < (1ull << 30) && mfma_h<kPoseidon2>(2) < (1ull << 30),
              "2^47 + sum of small weights * 2^32 stays below 2^63");

template <int HT, int M, int I>
__device__ __forceinline__ void add_earlier_small(uint64_t &L, uint64_t &H, const uint64_t *y)
{
    if constexpr (I < M) {
        constexpr uint64_t w = mfma_h<HT>(M - I);
        if constexpr (w < (1ull << 32)) {
            L = gl::vopaque64((uint64_t)gl::lo32(y[I]) * gl::opaque((uint32_t)w) + L);
            H = gl::vopaque64((uint64_t)gl::hi32(y[I]) * gl::opaque((uint32_t)w) + H);
        }
        add_earlier_small<HT, M, I + 1>(L, H, y);
    }
}

// x + w * y, lazy.  The sum added to the product's low word carries at most 1
// into the high word, and the total stays below (2^64 - 1)^2 + 2^64, so the
// high word plus the product's carry fits 64 bits.
__device__ __forceinline__ uint64_t mul_add_lazy(uint64_t y, uint64_t w, uint64_t x)
{
    uint64_t lo, hi, pc;
    gl::mul128c(y, w, lo, hi, pc);
    uint32_t c1, c2, c3, c4;
    const uint32_t l0 = __builtin_addc(gl::lo32(lo), gl::lo32(x), 0u, &c1);
    const uint32_t l1 = __builtin_addc(gl::hi32(lo), gl::hi32(x), c1, &c2);
    const uint32_t h0 = __builtin_addc(gl::lo32(hi), 0u, c2, &c3);
    const uint32_t h1 = __builtin_addc(gl::hi32(hi), 0u, c3, &c4);
    return gl::reduce128c_lazy(gl::pack(l0, l1), gl::pack(h0, h1), pc);
}

template <int HT, int M, int I>
__device__ __forceinline__ void add_earlier_large(uint64_t &x, const uint64_t *y)
{
    if constexpr (I < M) {
        constexpr uint64_t w = mfma_h<HT>(M - I);
        if constexpr (w >= (1ull << 32)) x = mul_add_lazy(y[I], w, x);
        add_earlier_large<HT, M, I + 1>(x, y);
    }
}

template <int HT, int M>
__device__ __forceinline__ uint64_t sbox_input(const uint32_t (&d)[4], const mfma::Pair &k, const uint64_t *y)
{
    uint64_t L = half_sum(d[0], d[1], k.l), H = half_sum(d[2], d[3], k.h);
    add_earlier_small<HT, M, 0>(L, H, y);
    uint64_t x = limb_combine(L, H);
    add_earlier_large<HT, M, 0>(x, y);
    return x;
}

// The S-box output of that input, in the wave forms of gl64.h.
template <int HT, int M>
__device__ __forceinline__ uint64_t sbox_output(const uint32_t (&d)[4], const mfma::Pair &k, const uint64_t *y)
{
    uint64_t L = half_sum(d[0], d[1], k.l), H = half_sum(d[2], d[3], k.h);
    add_earlier_small<HT, M, 0>(L, H, y);
    // the weights of earlier outputs widen the sum: top < 2^15 + their sum, and
    // a carry in one of 64 lanes once in 2^26 / top S-boxes
    if constexpr (mfma_h_sum<HT>(M) < (1ull << 21)) {
        uint64_t carry;
        const uint64_t x = limb_combine_rare(L, H, carry);
        return gl::pow7_wave(x, carry);
    }
    uint64_t x = limb_combine(L, H);
    add_earlier_large<HT, M, 0>(x, y);
    return gl::pow7_wave(x);
}

__device__ __forceinline__ void mfma_sboxes(uint64_t s[2][6])
{
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int e = 0; e < 6; e += 2) gl::pow7_wave2(s[t][e], s[t][e + 1]);
}

// This lane's slots 0..11 as B operands.
template <int NK>
__device__ __forceinline__ void mfma_state(mf_v4i (&b)[2][NK], const uint64_t s[2][6])
{
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int kappa = 0; kappa < 3; kappa++)
            b[t][kappa] = mfma_pair(mfma_bytes(s[t][2 * kappa]), mfma_bytes(s[t][2 * kappa + 1]));
}

// The permutation of 64 states (layout above); m: the work-group's tables.
// Lazy in and out.  All 64 lanes of the wave must be active.
template <int HT>
__device__ __forceinline__ void permute_mfma(uint64_t s[2][6], const MfmaLds &m)
{
    using namespace mfma;
    const uint32_t l = threadIdx.x & 63, h = l >> 5;
    // the tables through an offset the compiler cannot see through: operands
    // are read where they are used, not kept in registers across rounds
    auto tables = [&](const mf_v4i *&op, const uint64_t (*&row)[12][2]) {
        uint32_t lane = l, half = h;
        asm volatile("; tables %0 %1" : "+v"(lane), "+v"(half));
        op = &m.op[0][lane];
        row = reinterpret_cast<const uint64_t(*)[12][2]>(&m.row[0][6 * half][0]);
    };
    auto full_layer = [&](int r) {
        const mf_v4i *op;
        const uint64_t(*row)[12][2];
        tables(op, row);
        mf_v4i b[2][3];
        mfma_state(b, s);
        mfma_map<3>(s, b, op + 64 * kOpLayer, row[r]);
    };
    if constexpr (HT == kPoseidon) {
#pragma unroll
        for (int e = 0; e < 6; e++) {
            const uint64_t k = m.row[kRowFirst][6 * h + e][0];
#pragma unroll
            for (int t = 0; t < 2; t++) s[t][e] = gl::add(s[t][e], k);
        }
    } else {
        full_layer(kRowFirst);
    }
#pragma unroll 1
    for (int r = 0; r < 3; r++) {
        mfma_sboxes(s);
        full_layer(kRowFull + r);
    }
    mfma_sboxes(s);
    {  // full round 3's layer and partial rounds 4, 5
        const mf_v4i *op;
        const uint64_t(*row)[12][2];
        tables(op, row);
        const mf_v4i *eop = reinterpret_cast<const mf_v4i *>(c_mfma<HT>.op) + l;
        mf_v4i b3[2][3];
        mfma_state(b3, s);
        uint32_t x[2][2][4];
        mfma_outputs(x, b3, eop + 64 * kOpEntryX);
        uint64_t y[2];
        y[0] = sbox_output<HT, 0>(x[0][0], c_mfma<HT>.x_entry[0], y);
        y[1] = sbox_output<HT, 1>(x[1][0], c_mfma<HT>.x_entry[1], y);
        uint64_t y1 = mfma_bytes(y[0]), y2 = mfma_bytes(y[1]);
        swap_halves(y1, y2);
        mf_v4i b[2][4];
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
            for (int kappa = 0; kappa < 3; kappa++) b[t][kappa] = b3[t][kappa];
            b[t][3] = mfma_pair(t ? y2 : y1, 0);
        }
        mfma_map<4>(s, b, eop + 64 * kOpEntry, row[kRowEntry]);
    }
#pragma unroll 1
    for (int g = 0; g < kGroups; g++) {  // five partial rounds each
        const mf_v4i *op;
        const uint64_t(*row)[12][2];
        tables(op, row);
        mf_v4i b3[2][3];
        mfma_state(b3, s);
        uint32_t x[2][2][4];
        mfma_outputs(x, b3, op + 64 * kOpGroupX);
        // element 0 of permutation (h, j), and element 6 of both groups
        uint64_t x1 = s[0][0], e6 = s[1][0];
        swap_halves(x1, e6);
        const Pair *k = c_mfma<HT>.x_group[g];
        uint64_t y[5];
        y[0] = gl::pow7_wave(x1);
        y[1] = sbox_output<HT, 1>(x[0][0], k[0], y);
        y[2] = sbox_output<HT, 2>(x[0][1], k[1], y);
        y[3] = sbox_output<HT, 3>(x[1][0], k[2], y);
        y[4] = sbox_output<HT, 4>(x[1][1], k[3], y);
#pragma unroll
        for (int i = 0; i < 5; i++) y[i] = mfma_bytes(y[i]);
        e6 = mfma_bytes(e6);
        swap_halves(y[0], e6);    // slot 0: y_1 on half 0, element 6 on half 1
        swap_halves(y[1], y[3]);  // slots 12, 14
        swap_halves(y[2], y[4]);  // slots 13, 15
        mf_v4i b[2][4];
#pragma unroll
        for (int t = 0; t < 2; t++) {
#pragma unroll
            for (int kappa = 0; kappa < 3; kappa++) b[t][kappa] = b3[t][kappa];
            const uint64_t s0 = t ? e6 : y[0];
            b[t][0][0] = (int)gl::lo32(s0);
            b[t][0][1] = (int)gl::hi32(s0);
            b[t][3] = mfma_pair(t ? y[3] : y[1], t ? y[4] : y[2]);
        }
        mfma_map<4>(s, b, op + 64 * kOpGroup, row[kRowGroup + g]);
    }
#pragma unroll 1
    for (int r = 0; r < 4; r++) {
        mfma_sboxes(s);
        full_layer(kRowLast + r);
    }
}

}  // namespace zkx
