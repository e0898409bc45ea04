// The linear Merkle forest (layout: merkle_kernels.h) on 16 permutations per
// wave (poseidon_narrow.h), for Poseidon and Poseidon2 forests and levels too
// small to fill the chip with 64 per wave.
//
// A work-group of four waves owns a tile of 64 leaves, or of 128 nodes of a
// level that is already written (MerkleArgs::leaves null), hashes 16 leaves
// per wave and reduces the tile in LDS, 16 nodes per wave and step; tiles that
// stop below the caps go on through the arrival counters exactly as those of
// k_merkle_tile.  Every level costs one permutation's latency of this form
// (12 us) instead of a launch of its own at 64 per wave (35-45 us) or lane
// pairs and rows of 16 on the VALU (25-36 us).  The tables fill 62 KiB of LDS:
// two work-groups, two waves per SIMD (17 us per permutation).  Measured (one
// MI355X): forest of 2^13 leaves of 135, cap 4, 690 -> 325 us; 2^15 with
// Poseidon2 890 -> 500 us; commit of 20 x 2^10 rate 1 280 -> 167 us; the 11
// narrow levels of a 2^18 tree 480 -> 160 us.
#pragma once
#include "merkle_kernels.h"
#include "poseidon_narrow.h"

namespace zkx {

// v[up] without an index into registers.
__device__ __forceinline__ uint32_t pick(const uint32_t (&v)[kMerkleMaxPasses - 1], uint32_t up)
{
    static_assert(kMerkleMaxPasses == 4, "three upper passes");
    return up == 0 ? v[0] : up == 1 ? v[1] : v[2];
}

template <int HT>
__global__ void __launch_bounds__(kMerkleNarrowLanes) __attribute__((amdgpu_waves_per_eu(2)))
k_merkle_narrow(const MerkleArgs *__restrict__ jobs, uint32_t njobs, MerkleArgs one, uint32_t block0)
{
    constexpr uint32_t kTile = 1u << kMerkleNarrowNodesLog, kWaves = kMerkleNarrowLanes / 64;
    __shared__ uint64_t lds[kTile][4];
    __shared__ uint32_t lds_last;
    __shared__ NarrowLds tables;
    const uint32_t bid = blockIdx.x + block0;
    const MerkleArgs a = njobs ? *find_job(jobs, njobs, bid) : one;
    const uint32_t t = threadIdx.x, w = t >> 6, j = t & 15, q = (t >> 4) & 3;
    uint32_t up = 0;                  // upper passes done
    uint32_t cur = 1u << a.tile_log;  // nodes of this tile at the current level
    uint32_t lg_w = a.lg_w;           // log2 per-subtree width of the current level
    uint64_t first = ((uint64_t)bid - a.tile_begin) << a.tile_log;  // first node of the tile
    // digest element q of node g of the current level
    auto node = [&](uint64_t g) {
        return (lg_w ? node_ptr(a, g >> lg_w, lg_w, g & ((1ull << lg_w) - 1)) : gmem(a.cap) + 4 * g) + q;
    };

    narrow_fill<HT, kMerkleNarrowLanes>(tables);
    __syncthreads();
    const uint32_t n0 = 16 * w + j;  // this lane's node of the tile
    const bool have = n0 < cur;
    // the tile's nodes (of a level that is written) into LDS
    auto load_nodes = [&] {
#pragma unroll
        for (uint32_t n = 0; n < kTile; n += 16 * kWaves)
            if (n + n0 < cur) lds[n + n0][q] = *node(first + n + n0);
    };
    uint64_t s[3] = {0, 0, 0};
    if (!a.leaves) {
        load_nodes();
    } else if (16 * w < cur) {
        const uint32_t ls = a.leaf_size;
        const uint64_t leaf = first + n0;
        const gptr<const uint64_t> row = gmem(a.leaves) + (have ? leaf : first) * a.leaf_stride;
        const gptr<uint64_t> out = a.leaves_out && have ? gmem(a.leaves_out) + leaf * ls : nullptr;
        // this lane's elements idx + q and idx + 4 + q of a chunk, loaded one
        // permutation ahead
        auto load = [&](uint32_t idx, uint64_t (&v)[2]) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint32_t k = idx + 4 * u + q;
                if (k < ls) v[u] = row[(uint64_t)k * a.col_stride];
            }
        };
        uint64_t v[2] = {0, 0};
        load(0, v);
        for (uint32_t idx = 0; idx < ls; idx += 8) {
#pragma unroll
            for (int u = 0; u < 2; u++) {
                const uint32_t k = idx + 4 * u + q;
                if (k < ls) {
                    s[u] = v[u];
                    if (out) out[k] = v[u];
                }
            }
            if (ls <= 4) break;  // the elements themselves, zero-padded
            load(idx + 8, v);
            permute_narrow<HT>(s, tables);
        }
        if (ls > 4) s[0] = gl::canon(s[0]);
        if (have) {
            *node(leaf) = s[0];
            lds[n0][q] = s[0];
        }
    }
    if (lg_w == 0 || a.leaves_only) return;  // caps == leaves, or levels launched apart
    __syncthreads();

    while (true) {
        if (cur == 1) {
            // tile root: continue with the group's tile if this work-group is
            // the last of its group to get here (merkle_kernels.h)
            if (up >= a.n_next) return;
            const uint32_t tl = pick(a.next_tile_log, up), c0 = pick(a.next_ctr, up);
            const uint64_t grp = first >> tl;
            __threadfence();  // this tile's digests, before the arrival
            __syncthreads();
            if (t == 0) {
                uint32_t *c = a.ctr + c0 + grp;
                const bool last = atomicAdd(c, 1u) == (1u << tl) - 1;
                if (last) atomicExch(c, 0u);
                lds_last = last ? 1u : 0u;
            }
            __syncthreads();
            if (!lds_last) return;
            __threadfence();  // the other tiles' roots, after their arrivals
            up++;
            cur = 1u << tl;
            first = grp << tl;
            load_nodes();
            __syncthreads();
            continue;
        }
        // the level above: node n = hash of nodes 2n, 2n + 1 (state [l, r, 0])
        const uint32_t half = cur >> 1;
        static_assert(kTile / 2 <= 16 * kWaves, "one step per level");
        const bool busy = 16 * w < half, real = n0 < half;
        uint64_t x[3] = {0, 0, 0};
        if (busy) {
            if (real) {
                x[0] = lds[2 * n0][q];
                x[1] = lds[2 * n0 + 1][q];
            }
            permute_narrow<HT>(x, tables);
            x[0] = gl::canon(x[0]);
        }
        __syncthreads();
        lg_w -= 1;
        first >>= 1;
        if (real) {
            *node(first + n0) = x[0];
            lds[n0][q] = x[0];
        }
        if (lg_w == 0) return;  // the caps
        cur = half;
        __syncthreads();
    }
}

}  // namespace zkx
