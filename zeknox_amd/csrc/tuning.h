// Schedule parameters of one commit shape, and the per-device table the
// autotuner fills.  None of them changes a result: every setting computes
// the same LDE, digests and caps; they only change how the work is cut into
// launches and work-groups.
#pragma once
#include <stdint.h>

#include <tuple>

namespace zkx {

struct Tuning {
    // NTT: at most this many DIF stages per strided (column-interleaved)
    // pass, 1..9; the last pass takes up to 12 contiguous stages.
    uint32_t ntt_strided_max = 9;
    // NTT: 0 = strided passes as large as allowed and the rest in the last
    // pass; 1 = the stages spread evenly over the fewest passes.
    uint32_t ntt_even = 0;
    // Merkle: log2 lanes (leaves) per work-group tile, 8..10.
    uint32_t merkle_tile_log = 8;
    // Merkle, Poseidon leaves: 0 = the MDS layers of whole-wave leaf
    // permutations on the i8 matrix cores; 1 = every permutation on the VALU.
    uint32_t merkle_valu = 0;
    // Set by the caller (zkx_set_tuning): the schedule runs as it stands.
    // Otherwise (built-in default, autotuner) small Poseidon and Poseidon2
    // forests are built by the 16-permutations-per-wave kernel and transforms
    // of 2^13 to 2^20 in one or two launches where that is faster, and the
    // schedule is that of what is left to passes and tiles.
    bool by_caller = false;
};

// A commit shape: (columns, log2 degree, rate bits, hash type, leaf rows kept).
using TuneKey = std::tuple<uint32_t, uint32_t, uint32_t, uint32_t, bool>;

bool valid_tuning(const Tuning &t);

// Poseidon and Poseidon2 have a kernel with 16 permutations per wave
// (merkle_narrow.h) besides those with 64, for work whose time is one
// permutation's latency.
inline bool has_narrow_kernel(uint64_t hash_type) { return hash_type == 0 || hash_type == 3; }
// It builds forests of at most this many leaves (all trees of one hash in a
// launch) in one launch, all work-groups resident, two waves per SIMD.
// (135-element leaves, cap 4, in us, 64 / 16 per wave: Poseidon 2^13 690 /
// 325, 2^15 880 / 453, Poseidon2 2^15 890 / 502; 2^16 needs two rounds of the
// 16-per-wave waves, 590 us for the leaves against 580.)
constexpr uint64_t kNarrowLeaves = 1ull << 15;
// It finishes larger trees from the first level of at most this many children
// (over all trees of one hash): every tile of 128 is resident at once.
constexpr uint64_t kNarrowNodes = 1ull << 16;

// Keccak-256's trees finish in one launch of the leaf kernel, on tiles of 256
// nodes of a written level, from the same number of children: there a level
// is a permutation on a lane pair, 6 us, against 9.4 in a launch of its own.
// (Forest of 2^18 leaves of 135, cap 0, 484 -> 423 us; 2^20 1239 -> 1179.)
constexpr bool has_tile_top(uint64_t hash_type) { return hash_type == 1; }

// Whether one tree through the C-ABI Merkle entry points builds its levels
// with one launch per level (after a leaf-digests-only launch; Poseidon and
// Poseidon2 finish with one launch of the 16-per-wave kernel) rather than
// inside its leaf launch, given the device threshold `min_leaves` (default
// 2^20): Poseidon and Poseidon2 trees switch at min_leaves / 16, Keccak-256
// and Monolith at min_leaves / 4, Poseidon-BN128 at min_leaves / 32 (0:
// always).  Measured, fused against apart, 135-element leaves, cap 4, ms:
//   leaves  Poseidon      Poseidon2     Keccak-256     Monolith       Poseidon-BN128
//   2^13    0.324 / 0.639 0.362 / 0.679 0.164 / 0.166  0.490 / 0.479  33.6 / 31.1
//   2^15    0.449 / 0.679 0.498 / 0.725 0.185 / 0.189  0.540 / 0.534  36.6 / 33.6
//   2^16    0.792 / 0.717 0.917 / 0.767 0.194 / 0.200  0.556 / 0.555  38.4 / 35.3
//   2^17    0.957 / 0.882 1.083 / 0.941 0.270 / 0.265  0.698 / 0.699  49.4 / 46.5
//   2^18    1.62 / 1.48   1.77 / 1.58   0.429 / 0.394  1.078 / 1.060  75.9 / 72.6
//   2^19    3.13 / 2.84   3.50 / 3.00   0.931 / 0.661  2.071 / 1.763  146 / 129
//   2^20    6.13 / 5.32   6.74 / 5.70   1.720 / 1.160  3.645 / 3.148
// (Poseidon and Poseidon2 up to 2^15 against the 16-per-wave kernel.)
// Poseidon's and Poseidon2's narrow levels cost 12 us each in the 16-per-wave
// kernel against 25-36 us on lane pairs and rows inside the leaf launch, so
// every tree that is not built whole by that kernel gains.  Keccak's and
// Monolith's permutations are short, so what their fused trees' lower levels
// lose on ever fewer lanes weighs more (their line is left where both sides
// are within 2%).  Poseidon-BN128's levels are slow enough that a full-GPU
// launch per level pays at every size measured.
inline bool lone_tree_levels_apart(uint64_t num_leaves, uint64_t hash_type, uint64_t min_leaves)
{
    const uint32_t shift = hash_type == 2 ? 5 : has_narrow_kernel(hash_type) ? 4 : 2;
    return num_leaves >= (min_leaves >> shift);
}
// Whether the 16-per-wave kernel builds it whole: up to kNarrowLeaves, and
// below the line above.
inline bool lone_tree_narrow(uint64_t num_leaves, uint64_t hash_type, uint64_t min_leaves)
{
    return has_narrow_kernel(hash_type) && num_leaves <= kNarrowLeaves &&
           !lone_tree_levels_apart(num_leaves, hash_type, min_leaves);
}

// Work-group size (log2 lanes) of the C-ABI Merkle entry points for one tree of
// num_leaves leaves while the caller has not set a default schedule.
//
// Levels apart: the launch hashes leaves alone, and 2^8 lanes are as fast as any
// (135-element leaves, cap 4, one MI355X, ms, tiles 2^8 / 2^9 / 2^10: Poseidon
// 2^17 0.883 / 0.882 / 1.305, 2^20 5.28 / 5.30 / 5.36, Poseidon2 2^20 5.65 /
// 5.69 / 5.84, Keccak-256 2^20 1.180 / 1.198 / 1.284, Monolith 2^20 3.13 / 3.15 /
// 3.43).  Poseidon over BN254, either side of that by size (2^17 46.1 / 46.2 /
// 68.3, 2^18 73.8 / 76.1 / 72.5, 2^19 128 / 136 / 129, 2^20 234 / 256 / 241),
// keeps the sizes below.
//
// Levels inside the launch: a tree alone has no other tree's leaves to hide
// them, and they run at low occupancy at its end, so the largest tile that
// still gives every CU a work-group (2^lg / 2^tile >= 256) wins up to 2^18
// leaves.  Above, which takes a caller's threshold, leaves take several rounds
// of work-groups and 2^9 lanes win for Poseidon and Poseidon2, 2^8 for
// Keccak-256 and Monolith, 2^10 for Poseidon over BN254 (as measured; the
// cause is not analysed).  The same trees, fused:
//   Poseidon    2^16 0.79 / 0.91 / 1.39, 2^17 1.01 / 0.96 / 1.44,
//               2^18 1.74 / 1.66 / 1.63, 2^20 6.17 / 6.07 / 6.31;
//   Keccak-256  2^16 0.194 / 0.247 / 0.366, 2^17 0.293 / 0.269 / 0.388,
//               2^18 0.474 / 0.474 / 0.428, 2^20 1.72 / 1.75 / 1.71
//               (Poseidon2, Monolith alike);
//   BN254       2^14 35.3 / 42.5 / 66.4, 2^17 55 / 49 / 72, 2^18 100 / 92 / 76,
//               2^19 180 / 182 / 146.
// In a batch other trees' leaves hide that tail and the batch default or
// the autotuned schedule applies.  hash_type: merkle/merkle.h numbering.
inline uint32_t lone_tree_tile_log(uint64_t num_leaves, uint64_t hash_type, uint64_t min_leaves)
{
    const uint32_t lg = num_leaves ? 63u - (uint32_t)__builtin_clzll(num_leaves) : 0u;
    const bool bn254 = hash_type == 2;
    if (lg <= 16 || (!bn254 && lone_tree_levels_apart(num_leaves, hash_type, min_leaves))) return 8;
    if (lg <= 18) return lg - 8;
    if (bn254) return 10;
    return has_narrow_kernel(hash_type) ? 9 : 8;
}

// lone_tree_levels_apart for the forests of one hash in a batch of
// `batch_leaves` leaves in total (default threshold 2^18; Poseidon and
// Poseidon2 at an eighth).
// One commit of 135 x 2^13 / 2^14 / 2^15 rate 3 (2^16, 2^17, 2^18 leaves), and
// eight of 20 x 2^12 rate 3 (2^18 leaves), fused against apart, ms:
//   Poseidon    0.877 / 0.808   1.174 / 1.054   2.08 / 1.82   0.703 / 0.524
//   Poseidon2   1.004 / 0.858   1.347 / 1.120   2.38 / 2.00   0.806 / 0.572
//   Keccak-256  0.298 / 0.302   0.470 / 0.470   1.15 / 1.06   0.326 / 0.293
//   Monolith    0.658 / 0.660   0.940 / 0.892   1.61 / 1.44   0.523 / 0.472
inline bool batch_levels_apart(uint64_t batch_leaves, uint64_t hash_type, uint64_t min_leaves)
{
    return batch_leaves > 0 && batch_leaves >= (has_narrow_kernel(hash_type) ? min_leaves >> 3 : min_leaves);
}
// Whether the 16-per-wave kernel builds a hash's forests of a batch
// (hash_leaves in all) whole: up to kNarrowLeaves, and below a quarter of
// min_leaves, which is above them by default.
inline bool batch_narrow(uint64_t hash_leaves, uint64_t hash_type, uint64_t min_leaves)
{
    return has_narrow_kernel(hash_type) && hash_leaves <= kNarrowLeaves && hash_leaves < (min_leaves >> 2);
}

}  // namespace zkx
