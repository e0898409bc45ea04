// Poseidon and Poseidon2 with 16 permutations per wave, four lanes each: for
// trees, levels and batches too small to fill the chip, whose time is one
// permutation's latency (poseidon_mfma.h's form runs 64 per wave).
//
// The maps are those of poseidon_mfma.h on v_mfma_i32_16x16x64_i8, which
// computes D[i][j] = sum_{q, n} A_{16q+i}[n] * B_{16q+j}[n] over the 16 bytes n
// each lane supplies; lane 16q' + j receives D[4q' + r][j] in its register r.
// Lane l (column j = l & 15, lane group q = l >> 4) holds the elements q,
// 4 + q, 8 + q of permutation j, and the S-box outputs of the partial rounds
// enter through a fourth slot.  The S-box inputs x_j of a group of partial
// rounds are outputs for every lane group alike, so all four run the serial
// chain of S-boxes and no lane waits for another's.
//
// Bound: one wave alone on a SIMD issues a multiply-add or a carry every 5.4
// cycles and a plain 32-bit operation every 4 (measured), and waits out what
// nothing covers, so the latency is the wave's instruction count.  A full
// round is 3 S-boxes per lane instead of 12, a partial round one; 64 per wave
// takes 34 us per permutation of a lone wave, this form 11.6.  (The products
// with a rare borrow of the 64-per-wave form lose here: a lone wave waits out
// their branches, 324 -> 340 us for a forest of 2^13 leaves of 135.)
#pragma once
#include "poseidon_mfma.h"

namespace zkx {

template <int HT>
__device__ const mfma::NarrowTables c_narrow = mfma::make_narrow<HT>();

// What a work-group keeps of the tables in LDS.
struct NarrowLds {
    mf_v4i op[mfma::kNarrowOps][64];
    alignas(16) uint64_t row[mfma::kRows][12][2];
};

template <int HT, int N>
__device__ __forceinline__ void narrow_fill(NarrowLds &m)
{
    copy_to_lds<mfma::kNarrowOps * 64, N>(&m.op[0][0], reinterpret_cast<const mf_v4i *>(c_narrow<HT>.op));
    copy_to_lds<mfma::kRows * 12, N>(reinterpret_cast<mf_v4i *>(m.row), reinterpret_cast<const mf_v4i *>(c_mfma<HT>.row));
}

// Lane group 0's x on every lane group (permlane swaps: poseidon_mfma.h).
__device__ __forceinline__ uint64_t from_group0(uint64_t x)
{
    uint32_t a0 = gl::lo32(x), a1 = gl::hi32(x), b0, b1;
    asm("v_mov_b32 %[b0], %[a0]\n\t"
        "v_mov_b32 %[b1], %[a1]\n\t"
        "s_nop 1\n\t"
        "v_permlane32_swap_b32 %[a0], %[b0]\n\t"
        "v_permlane32_swap_b32 %[a1], %[b1]\n\t"
        "s_nop 1\n\t"
        "v_mov_b32 %[b0], %[a0]\n\t"
        "v_mov_b32 %[b1], %[a1]\n\t"
        "s_nop 1\n\t"
        "v_permlane16_swap_b32 %[a0], %[b0]\n\t"
        "v_permlane16_swap_b32 %[a1], %[b1]"
        : [a0] "+v"(a0), [a1] "+v"(a1), [b0] "=&v"(b0), [b1] "=&v"(b1));
    return gl::pack(a0, a1);
}

// m ? a : b for m all ones or zero.
__device__ __forceinline__ uint64_t pick(uint32_t m, uint64_t a, uint64_t b)
{
    const uint64_t mm = gl::pack(m, m);
    return (a & mm) | (b & ~mm);
}

// One wave alone hides nothing: what follows issues each phase's MFMAs and
// LDS reads ahead of vector work that does not need them, and keeps the
// compiler from moving them back to their uses.
__device__ __forceinline__ void phase_end() { __builtin_amdgcn_sched_barrier(0); }

// The operands of one map in registers: [M-block][K-chunk].
template <int NB>
struct NarrowOps {
    mf_v4i a[NB][2];
    __device__ __forceinline__ explicit NarrowOps(const mf_v4i *op)
    {
#pragma unroll
        for (int i = 0; i < 2 * NB; i++) a[i / 2][i % 2] = op[64 * i];
    }
    // keeps them until p, computed from the sums, is there (hold_operands)
    __device__ __forceinline__ void hold(uint32_t p) const
    {
#pragma unroll
        for (int i = 0; i < 2 * NB; i++) asm volatile("; hold %0 %1" ::"v"(p), "v"(a[i / 2][i % 2]));
    }
};

// Digit sums of a map: K-chunk 0 (slots 0, 1), then K-chunk 1.
template <int NB>
struct NarrowSums {
    mf_v4i d[NB];
    __device__ __forceinline__ void first(const NarrowOps<NB> &o, const mf_v4i &b)
    {
#pragma unroll
        for (int i = 0; i < NB; i++) d[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a[i][0], b, mf_v4i{}, 0, 0, 0);
    }
    __device__ __forceinline__ void second(const NarrowOps<NB> &o, const mf_v4i &b)
    {
#pragma unroll
        for (int i = 0; i < NB; i++) d[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(o.a[i][1], b, d[i], 0, 0, 0);
    }
    // the digit pairs of output o (M-blocks 2o, 2o + 1)
    __device__ __forceinline__ void pairs(int o, uint32_t (&p)[4]) const
    {
#pragma unroll
        for (int n = 0; n < 4; n++) p[n] = digit_pair(d[2 * o + n / 2][2 * (n % 2)], d[2 * o + n / 2][2 * (n % 2) + 1]);
    }
};

// The same for a map's slots.
__device__ __forceinline__ void hold_slots(const mf_v4i &b, uint32_t p) { asm volatile("; hold %0 %1" ::"v"(p), "v"(b)); }

// A lane's three constants of one row.
struct NarrowRow {
    uint64_t l[3], h[3];
    __device__ __forceinline__ explicit NarrowRow(const uint64_t (*row)[2])
    {
#pragma unroll
        for (int a = 0; a < 3; a++) {
            l[a] = row[4 * a][0];
            h[a] = row[4 * a][1];
        }
    }
};

// s <- the recombined map; o, b0, b1: the operands and slots it was given.
__device__ __forceinline__ void narrow_state(uint64_t (&s)[3], const NarrowSums<6> &sum, const NarrowRow &k,
                                             const NarrowOps<6> &o, const mf_v4i &b0, const mf_v4i &b1)
{
#pragma unroll
    for (int a = 0; a < 3; a++) {
        uint32_t p[4];
        sum.pairs(a, p);
        if (a == 2) {
            hold_slots(b0, p[3]);
            hold_slots(b1, p[3]);
            o.hold(p[3]);
        }
        s[a] = limb_combine(half_sum(p[0], p[1], k.l[a]), half_sum(p[2], p[3], k.h[a]));
    }
}

// The permutation of 16 states (layout above).  Lazy in and out.  All 64
// lanes of the wave must be active.
template <int HT>
__device__ __forceinline__ void permute_narrow(uint64_t (&s)[3], const NarrowLds &m)
{
    using namespace mfma;
    const uint32_t l = threadIdx.x & 63, q = l >> 4;
    const uint32_t odd = 0u - (q & 1), upper = 0u - (q >> 1), group0 = ~(odd | upper);
    const mf_v4i *op = &m.op[0][l];
    auto row = [&](int r) { return reinterpret_cast<const uint64_t(*)[2]>(&m.row[r][q][0]); };
    auto slots01 = [&] { return mfma_pair(mfma_bytes(s[0]), mfma_bytes(s[1])); };
    auto slots23 = [&](uint64_t s3) { return mfma_pair(mfma_bytes(s[2]), s3); };
    // a layer with the S-boxes before it (`sboxes`): the sums of slots 0 and 1
    // run beside the third S-box
    auto full_layer = [&](const NarrowOps<6> &o, int r, bool sboxes) {
        const NarrowRow k(row(r));
        NarrowSums<6> sum;
        if (sboxes) gl::pow7_lazy2(s[0], s[1]);
        const mf_v4i b0 = slots01();
        sum.first(o, b0);
        phase_end();
        if (sboxes) s[2] = gl::pow7_lazy(s[2]);
        const mf_v4i b1 = slots23(0);
        sum.second(o, b1);
        phase_end();
        narrow_state(s, sum, k, o, b0, b1);
    };
    {
        const NarrowOps<6> o(op + 64 * kNarrowLayer);
        if constexpr (HT == kPoseidon) {
#pragma unroll
            for (int a = 0; a < 3; a++) s[a] = gl::add(s[a], row(kRowFirst)[4 * a][0]);
        } else {
            full_layer(o, kRowFirst, false);
        }
#pragma unroll 1
        for (int r = 0; r < 3; r++) full_layer(o, kRowFull + r, true);
    }
    {  // full round 3's S-boxes and layer, partial rounds 4, 5
        const NarrowOps<4> ox(op + 64 * kNarrowEntryX);
        const NarrowOps<6> o(op + 64 * kNarrowEntry);
        const NarrowRow k(row(kRowEntry));
        phase_end();
        gl::pow7_lazy2(s[0], s[1]);
        const mf_v4i b0 = slots01();
        NarrowSums<4> sx;
        NarrowSums<6> sum;
        sx.first(ox, b0);
        sum.first(o, b0);
        phase_end();
        s[2] = gl::pow7_lazy(s[2]);
        const mf_v4i bx = slots23(0);
        sx.second(ox, bx);
        phase_end();
        uint32_t x[2][4];
        sx.pairs(0, x[0]);
        sx.pairs(1, x[1]);
        hold_slots(bx, x[1][3]);
        ox.hold(x[1][3]);
        uint64_t y[2];
        y[0] = gl::pow7_lazy(sbox_input<HT, 0>(x[0], c_mfma<HT>.x_entry[0], y));
        y[1] = gl::pow7_lazy(sbox_input<HT, 1>(x[1], c_mfma<HT>.x_entry[1], y));
        const mf_v4i b1 = slots23(mfma_bytes(pick(upper, y[1], y[0])));
        sum.second(o, b1);
        phase_end();
        narrow_state(s, sum, k, o, b0, b1);
    }
    {
        const NarrowOps<8> ox(op + 64 * kNarrowGroupX);
        const NarrowOps<6> o(op + 64 * kNarrowGroup);
#pragma unroll 1
        for (int g = 0; g < kGroups; g++) {  // five partial rounds each
            const NarrowRow k(row(kRowGroup + g));
            const Pair *kx = c_mfma<HT>.x_group[g];
            const mf_v4i bx0 = slots01(), bx1 = slots23(0);
            NarrowSums<8> sx;
            NarrowSums<6> sum;
            sx.first(ox, bx0);
            sx.second(ox, bx1);
            phase_end();
            uint64_t y[5];
            y[0] = gl::pow7_lazy(from_group0(s[0]));
            // slot 0 of lane group 0: y_1; the fourth slot of group q: y_{q + 2}
            const mf_v4i b0 = mfma_pair(mfma_bytes(pick(group0, y[0], s[0])), mfma_bytes(s[1]));
            sum.first(o, b0);
            phase_end();
            uint32_t x[4][4];
#pragma unroll
            for (int i = 0; i < 4; i++) sx.pairs(i, x[i]);
            hold_slots(bx0, x[3][3]);
            hold_slots(bx1, x[3][3]);
            ox.hold(x[3][3]);
            y[1] = gl::pow7_lazy(sbox_input<HT, 1>(x[0], kx[0], y));
            y[2] = gl::pow7_lazy(sbox_input<HT, 2>(x[1], kx[1], y));
            y[3] = gl::pow7_lazy(sbox_input<HT, 3>(x[2], kx[2], y));
            y[4] = gl::pow7_lazy(sbox_input<HT, 4>(x[3], kx[3], y));
            const mf_v4i b1 = slots23(mfma_bytes(pick(upper, pick(odd, y[4], y[3]), pick(odd, y[2], y[1]))));
            sum.second(o, b1);
            phase_end();
            narrow_state(s, sum, k, o, b0, b1);
        }
    }
    {
        const NarrowOps<6> o(op + 64 * kNarrowLayer);
#pragma unroll 1
        for (int r = 0; r < 4; r++) full_layer(o, kRowLast + r, true);
    }
}

}  // namespace zkx
