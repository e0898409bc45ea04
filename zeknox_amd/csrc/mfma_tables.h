// Compile-time tables of the matrix-core Poseidon and Poseidon2 permutations
// (poseidon_mfma.h: 64 per wave; poseidon_narrow.h: 16 per wave): the linear
// maps between S-boxes, cut into signed bytes as operands of
// v_mfma_i32_32x32x32_i8 and v_mfma_i32_16x16x64_i8, and their folded
// constants.
//
// Both permutations are 8 full rounds and 22 partial rounds of x^7 with a
// linear layer after each round (poseidon/poseidon.cu:563-838,
// poseidon2/poseidon2.cu:65-209).  Between full rounds the map is the layer
// itself.  The partial rounds touch one element each, so k of them in a row
// are one linear map with k S-boxes inside: with t the state before the
// first of them (round constants added) and y_1..y_k the S-box outputs,
//   x_1 = t_0,   x_j = L_j(t_1..t_11) + sum_{i<j} h_{j-i} y_i + const,
//   y_j = x_j^7, state after = F(t_1..t_11, y_1..y_k) + const,
// with h_m the weight with which an S-box output reaches element 0 m layers
// later through elements 1..11.  The 22 partial rounds run as an entry map
// (the layer of full round 3 and rounds 4, 5: two S-boxes) and four groups
// of five rounds.  L, F and the constants come from iterating the layers on
// affine forms over the slots below.
//
// Slots.  A map reads 16 slots of 64 bits: slots 0..11 the state elements
// (slot 0: y_1 in a group), slots 12..15 further S-box outputs (a group:
// y_2..y_5; the entry: y_1 in 12, y_2 in 14).  64 per wave: K-chunk kappa of
// 32 bytes holds the slots 6h + 2 kappa + {0, 1} of lane half h for
// kappa < 3, and 12 + 2h + {0, 1} for kappa = 3.  16 per wave: K-chunk kappa
// of 64 bytes holds the slots 8 kappa + q and 8 kappa + 4 + q of lane group q.
//
// Bytes.  A coefficient c applied to byte b of a slot contributes
// c * 2^(8b) mod p, written in eight signed digits of base 256: one output
// row per (output element, digit), one column per (slot, byte).  So a map
// with any coefficients mod p costs the same products as the small
// circulant itself.  The state's bytes enter as u - 128, which the constants
// put right: the bytes' 128s add 0x8080808080808080 * sum of coefficients.
#pragma once
#include "gl64.h"
#include "gl_constants.h"
#include "merkle_types.h"

namespace zkx {
namespace mfma {

// Operands of 64 lanes x 16 bytes, in the order [M-block beta][K-chunk kappa].
constexpr int kOpLayer = 0;    // 9: the full rounds' layer
constexpr int kOpGroup = 9;    // 12: F of five partial rounds
constexpr int kOpGroupX = 21;  // 3: x_2..x_5 of five partial rounds
constexpr int kOpsLds = 24;    // the operands above are used often: kept in LDS
constexpr int kOpEntry = 24;   // 12: F of the entry map
constexpr int kOpEntryX = 36;  // 3: x_1, x_2 of the entry map
constexpr int kOps = 39;

// Constant rows, added by the map that they are named after.
constexpr int kRowFirst = 0;   // Poseidon: the first round's constants as they are; Poseidon2: the first layer
constexpr int kRowFull = 1;    // 3: full rounds 0..2
constexpr int kRowEntry = 4;   // entry map
constexpr int kRowGroup = 5;   // 4: groups of partial rounds
constexpr int kRowLast = 9;    // 4: full rounds 26..29
constexpr int kRows = 13;

constexpr int kGroups = 4, kGroupRounds = 5, kEntryRounds = 2;

// A constant as two addends of the recombination: value = l + 2^32 h (mod p).
struct Pair {
    uint64_t l, h;
};

struct Tables {
    alignas(16) uint8_t op[kOps][64][16];
    alignas(16) Pair row[kRows][12];
    Pair x_entry[2];         // constants of x_1, x_2 of the entry map
    Pair x_group[kGroups][4];  // constants of x_2..x_5 of each group
};

// Operands of the 16-per-wave form, in the order [M-block][K-chunk of 2]: M-
// block 2a + n holds digits 4n..4n + 3 of element 4a + q for lane group q, or
// of output a for every lane group.
constexpr int kNarrowLayer = 0;    // 12: the full rounds' layer
constexpr int kNarrowGroup = 12;   // 12: F of five partial rounds
constexpr int kNarrowGroupX = 24;  // 16: x_2..x_5
constexpr int kNarrowEntry = 40;   // 12: F of the entry map
constexpr int kNarrowEntryX = 52;  // 8: x_1, x_2
constexpr int kNarrowOps = 60;

struct NarrowTables {
    alignas(16) uint8_t op[kNarrowOps][64][16];
};

constexpr uint64_t cadd(uint64_t a, uint64_t b)
{
    const unsigned __int128 s = (unsigned __int128)a + b;
    return (uint64_t)(s >= gl::P ? s - gl::P : s);
}
constexpr uint64_t csub(uint64_t a, uint64_t b) { return a >= b ? a - b : a + (gl::P - b); }

constexpr uint64_t kRcPoseidon[30 * 12] = {ZK_POSEIDON_RC_LIST};
constexpr uint64_t kRcPoseidon2[30 * 12] = {ZK_POSEIDON2_RC_LIST};
constexpr uint64_t kCirc[12] = {ZK_POSEIDON_MDS_CIRC_LIST};
constexpr uint64_t kDiag[12] = {ZK_POSEIDON_MDS_DIAG_LIST};
constexpr uint64_t kDiag2[12] = {ZK_POSEIDON2_DIAG_LIST};
constexpr uint64_t kM4[4][4] = {{5, 7, 1, 3}, {4, 6, 1, 1}, {1, 3, 5, 7}, {1, 1, 4, 6}};

// Layer coefficient (row r, column c) after a full or a partial round.
template <int HT>
constexpr uint64_t layer(int r, int c, bool partial)
{
    if (HT == kPoseidon) return kCirc[(c - r + 12) % 12] + (r == c ? kDiag[r] : 0);
    if (partial) return r == c ? cadd(kDiag2[r], 1) : 1;
    return kM4[r % 4][c % 4] * (r / 4 == c / 4 ? 2 : 1);
}

// Constant added to element i before the S-boxes of round r (30: none).
template <int HT>
constexpr uint64_t round_constant(int r, int i)
{
    if (r >= 30) return 0;
    if (HT == kPoseidon) return kRcPoseidon[12 * r + i];
    return r >= 4 && r < 26 && i > 0 ? 0 : kRcPoseidon2[12 * r + i];
}

// An affine form over the 16 slots.
struct Form {
    uint64_t c[16] = {}, k = 0;
};
struct State {
    Form e[12];
};

// The state after one more layer, with the constants of round r added.
template <int HT>
constexpr State step(const State &v, bool partial, int r)
{
    State out;
    for (int i = 0; i < 12; i++) {
        for (int j = 0; j < 12; j++) {
            const uint64_t m = layer<HT>(i, j, partial);
            for (int q = 0; q < 16; q++)
                if (v.e[j].c[q]) out.e[i].c[q] = cadd(out.e[i].c[q], gl::cmul(m, v.e[j].c[q]));
            if (v.e[j].k) out.e[i].k = cadd(out.e[i].k, gl::cmul(m, v.e[j].k));
        }
        out.e[i].k = cadd(out.e[i].k, round_constant<HT>(r, i));
    }
    return out;
}

constexpr Form slot(int q)
{
    Form f;
    f.c[q] = 1;
    return f;
}

constexpr State identity()
{
    State v;
    for (int i = 0; i < 12; i++) v.e[i] = slot(i);
    return v;
}

// Eight signed digits of base 256 of a representative of v mod p.
constexpr void digits(uint64_t v, int (&d)[8])
{
    // above 0x7f..7f the digits would carry out: v - p instead
    __int128 x = (__int128)v - (v > 0x7f7f7f7f7f7f7f7full ? (__int128)gl::P : 0);
    for (int i = 0; i < 8; i++) {
        int t = (int)(x & 255);
        if (t > 127) t -= 256;
        d[i] = t;
        x = (x - t) / 256;
    }
}

// Bias of each half of a constant pair: the recombined digit sums of one half
// are at most 128 products of 128 * 128 in four digits, below 2^45.1.
constexpr uint64_t kBias = 1ull << 46;

// The constant of a form as an addend pair, with the bytes' 128s and the bias
// (kBias * (1 + 2^32)) put right.  `used`: the slots that the map reads.
constexpr Pair addend(const Form &f, uint32_t used)
{
    uint64_t sum = 0;
    for (int q = 0; q < 16; q++)
        if (used >> q & 1) sum = cadd(sum, f.c[q]);
    uint64_t t = cadd(f.k, gl::cmul(0x8080808080808080ull, sum));
    t = csub(t, cadd(kBias, gl::cmul(kBias, 1ull << 32)));
    return Pair{kBias + (uint32_t)t, kBias + (t >> 32)};
}

// Rows of the operands from `op` on: M-block beta holds output elements
// 6h' + 2 beta + {0, 1} of lane half h' (nblocks == 3), or outputs
// 2h' + {0, 1} (one block).
constexpr void put(Tables &t, int op, int nblocks, int nchunks, const Form *rows, int nrows)
{
    for (int R = 0; R < nrows; R++) {
        const int hp = nblocks == 3 ? R / 6 : R / 2, e = nblocks == 3 ? R % 6 : R % 2;
        for (int q = 0; q < (nchunks == 4 ? 16 : 12); q++) {
            const int kappa = q < 12 ? q % 6 / 2 : 3, ha = q < 12 ? q / 6 : (q - 12) / 2;
            uint64_t v = rows[R].c[q];
            if (!v) continue;
            for (int b = 0; b < 8; b++) {
                int d[8] = {};
                digits(v, d);
                for (int n = 0; n < 8; n++) {
                    const int i = 8 * (2 * (e % 2) + n / 4) + 4 * hp + n % 4;  // row of the M-block
                    t.op[op + (e / 2) * nchunks + kappa][32 * ha + i][8 * (q % 2) + b] = (uint8_t)d[n];
                }
                v = gl::cmul(v, 256);
            }
        }
    }
}

// h_1..h_4 (h_m: an S-box output's weight in the S-box input m rounds on).
struct Weights {
    uint64_t v[kGroupRounds];
};
template <int HT>
constexpr Weights partial_weights()
{
    Weights w{};
    State v = identity();
    for (int m = 1; m < kGroupRounds; m++) {
        v = step<HT>(v, true, 30);
        w.v[m] = v.e[0].c[0];
        v.e[0] = slot(12);
    }
    return w;
}

// Rows of the 16-per-wave operands from `op` on.
constexpr void put_narrow(NarrowTables &t, int op, const Form *rows, int nrows, bool every_group)
{
    for (int R = 0; R < nrows; R++)
        for (int q = 0; q < 16; q++) {
            uint64_t v = rows[R].c[q];
            if (!v) continue;
            for (int b = 0; b < 8; b++) {
                int d[8] = {};
                digits(v, d);
                for (int n = 0; n < 8; n++) {
                    const int block = 2 * (every_group ? R : R / 4) + n / 4;
                    for (int g = every_group ? 0 : R % 4; g <= (every_group ? 3 : R % 4); g++)
                        t.op[op + 2 * block + q / 8][16 * (q % 4) + 4 * g + n % 4][8 * (q / 4 % 2) + b] = (uint8_t)d[n];
                }
                v = gl::cmul(v, 256);
            }
        }
}

constexpr uint32_t kState = 0x0FFF, kAll = 0xFFFF;

// The maps as affine forms: what the operands and constants are made of.
struct Maps {
    State full;               // the full rounds' layer, without constants
    State entry;              // the layer of full round 3, then partial rounds 4 and 5
    Form x_entry[2];          // x_1, x_2
    State group[kGroups];     // five partial rounds
    Form x_group[kGroups][4];  // x_2..x_5, their y terms left out
};

constexpr Form of_state(Form f, int first)
{
    for (int q = 0; q < 16; q++)
        if (q < first || q >= 12) f.c[q] = 0;
    return f;
}

template <int HT>
constexpr Maps maps()
{
    Maps m{};
    m.full = step<HT>(identity(), false, 30);
    m.entry = identity();
    for (int j = 0; j <= kEntryRounds; j++) {
        m.entry = step<HT>(m.entry, j > 0, 4 + j);
        if (j == kEntryRounds) break;
        m.x_entry[j] = of_state(m.entry.e[0], 0);  // x_2's y_1 term: h_1
        m.entry.e[0] = slot(12 + 2 * j);
    }
    for (int g = 0; g < kGroups; g++) {
        State &v = m.group[g];
        v = identity();  // slot 0: y_1
        for (int j = 0; j < kGroupRounds; j++) {
            v = step<HT>(v, true, 4 + kEntryRounds + kGroupRounds * g + j + 1);
            if (j == kGroupRounds - 1) break;
            m.x_group[g][j] = of_state(v.e[0], 1);
            v.e[0] = slot(12 + j);
        }
    }
    return m;
}

template <int HT>
constexpr Tables make()
{
    Tables t{};
    Maps m = maps<HT>();
    put(t, kOpLayer, 3, 3, m.full.e, 12);
    for (int i = 0; i < 12; i++) {
        if (HT == kPoseidon) t.row[kRowFirst][i] = Pair{round_constant<HT>(0, i), 0};
        auto row = [&](int at, int r) {
            m.full.e[i].k = round_constant<HT>(r, i);
            t.row[at][i] = addend(m.full.e[i], kState);
        };
        if (HT != kPoseidon) row(kRowFirst, 0);
        for (int r = 0; r < 3; r++) row(kRowFull + r, r + 1);
        for (int r = 0; r < 4; r++) row(kRowLast + r, r + 27);
        t.row[kRowEntry][i] = addend(m.entry.e[i], kAll);
        for (int g = 0; g < kGroups; g++) t.row[kRowGroup + g][i] = addend(m.group[g].e[i], kAll);
    }
    const Form xe[4] = {m.x_entry[0], Form{}, m.x_entry[1], Form{}};  // x_1 on half 0, x_2 on half 1
    put(t, kOpEntryX, 1, 3, xe, 4);
    put(t, kOpEntry, 3, 4, m.entry.e, 12);
    put(t, kOpGroupX, 1, 3, m.x_group[0], 4);
    put(t, kOpGroup, 3, 4, m.group[0].e, 12);
    for (int j = 0; j < kEntryRounds; j++) t.x_entry[j] = addend(m.x_entry[j], kState);
    for (int g = 0; g < kGroups; g++)
        for (int j = 0; j < 4; j++) t.x_group[g][j] = addend(m.x_group[g][j], kState);
    return t;
}

template <int HT>
constexpr NarrowTables make_narrow()
{
    NarrowTables t{};
    const Maps m = maps<HT>();
    put_narrow(t, kNarrowLayer, m.full.e, 12, false);
    put_narrow(t, kNarrowGroup, m.group[0].e, 12, false);
    put_narrow(t, kNarrowGroupX, m.x_group[0], 4, true);
    put_narrow(t, kNarrowEntry, m.entry.e, 12, false);
    put_narrow(t, kNarrowEntryX, m.x_entry, kEntryRounds, true);
    return t;
}

}  // namespace mfma
}  // namespace zkx
