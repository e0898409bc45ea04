// Host side of the Merkle forest: argument checks mirroring merkle.cpp:19-124
// and merkle.cu:165-244, the pass schedule of merkle_kernels.h, and launches
// of pass lists (one tree, or many trees of a commit batch).
#include "merkle.h"

#include <algorithm>
#include <string>

#include "merkle_launch.h"

namespace zkx {

namespace {

bool is_pow2(uint64_t x) { return x && !(x & (x - 1)); }
uint32_t log2u(uint64_t x) { return 63 - __builtin_clzll(x); }

}  // namespace

void check_merkle(const MerkleSpec &s)
{
    if (s.hash_type > kMonolith)
        invalid("hash type " + std::to_string(s.hash_type) +
                " is not provided (Poseidon 0, Keccak 1, Poseidon-BN128 2, Poseidon2 3, Monolith 4)");
    if (!s.caps || !s.leaves) invalid("null cap or leaf buffer");
    if (!is_pow2(s.num_leaves) || !is_pow2(s.num_caps) || s.num_caps > s.num_leaves)
        invalid("leaves and caps must be powers of two with caps <= leaves");
    // (the sponges of eight elements a block count them in steps of eight in 32
    // bits: beyond 2^32 - 8 the count would wrap and never end)
    if (s.leaf_size == 0 || s.leaf_size > (s.hash_type == kKeccak ? 0xFFFFFFFFull : 0xFFFFFFF8ull))
        invalid("leaf size out of range");
    if (s.num_caps == s.num_leaves) return;
    if ((1ull << s.cap_height) != s.num_caps) invalid("cap_buf_size must be 2^cap_height");
    if (s.num_digests != 2 * (s.num_leaves - s.num_caps))
        invalid("digests_buf_size must be 2 * (leaves_buf_size - cap_buf_size)");
    if (!s.digests) invalid("null digest buffer");
}

// Passes from the level of width 2^lg_w per subtree up, in tiles of at most
// 2^tile_log_max nodes, those above the first pass of 2^upper_log_max.
static uint32_t plan_passes(const MerkleSpec &s, MerkleArgs (&passes)[kMerkleMaxPasses], uint32_t tile_log_max,
                            uint32_t upper_log_max, uint32_t lg_w)
{
    MerkleArgs a{};
    a.leaves = s.leaves;
    a.leaves_out = s.leaves_out;
    a.dig = s.digests;
    a.cap = s.caps;
    a.leaf_size = (uint32_t)s.leaf_size;
    a.leaf_stride = s.leaf_stride;
    a.col_stride = s.col_stride;
    a.leaf_valu = s.leaf_valu;
    if (s.num_caps == s.num_leaves) {
        a.count = s.num_leaves;
        a.lg_w = 0;
        a.tile_log = std::min<uint32_t>(tile_log_max, log2u(a.count));
        passes[0] = a;
        return 1;
    }
    const uint32_t h = log2u(s.num_caps);
    a.sdl = s.num_digests >> h;
    uint32_t n = 0;
    while (true) {
        if (n == (uint32_t)kMerkleMaxPasses) invalid("tree too large");
        a.count = s.num_caps << lg_w;
        a.lg_w = lg_w;
        a.tile_log = std::min<uint32_t>(n ? upper_log_max : tile_log_max, log2u(a.count));
        passes[n++] = a;
        if (lg_w <= a.tile_log) break;  // this pass reaches the caps
        lg_w -= a.tile_log;
    }
    return n;
}

uint32_t plan_merkle(const MerkleSpec &s, MerkleArgs (&passes)[kMerkleMaxPasses], uint32_t tile_log_max)
{
    if (tile_log_max < (uint32_t)kMerkleMinTileLog || tile_log_max > (uint32_t)kMerkleMaxTileLog)
        invalid("Merkle tile size out of range");
    return plan_passes(s, passes, tile_log_max, tile_log_max, log2u(s.num_leaves) - log2u(s.num_caps));
}

uint64_t plan_merkle_narrow(const MerkleSpec &s, const uint32_t *written, MerkleArgs &out)
{
    MerkleArgs passes[kMerkleMaxPasses];
    const uint32_t nodes_log = has_tile_top(s.hash_type) ? kMerkleMinTileLog : kMerkleNarrowNodesLog;
    const uint32_t n = plan_passes(s, passes, written ? nodes_log : kMerkleNarrowTileLog, nodes_log,
                                   written ? *written : log2u(s.num_leaves) - log2u(s.num_caps));
    if (written) passes[0].leaves = nullptr;
    return fuse_merkle_passes(passes, n, out);
}

void plan_merkle(const MerkleSpec &s, std::vector<MerkleArgs> &passes, uint32_t tile_log_max)
{
    MerkleArgs p[kMerkleMaxPasses];
    const uint32_t n = plan_merkle(s, p, tile_log_max);
    passes.insert(passes.end(), p, p + n);
}

uint64_t fuse_merkle_passes(const MerkleArgs *passes, uint32_t n, MerkleArgs &out)
{
    if (n == 0 || n > (uint32_t)kMerkleMaxPasses) invalid("internal: Merkle pass plan");
    out = passes[0];
    out.n_next = n - 1;
    out.ctr = nullptr;
    uint64_t ctrs = 0;
    for (uint32_t p = 1; p < n; p++) {
        out.next_tile_log[p - 1] = passes[p].tile_log;
        out.next_ctr[p - 1] = (uint32_t)ctrs;
        ctrs += passes[p].count >> passes[p].tile_log;
    }
    if (ctrs > 0xFFFFFFFFull) invalid("tree too large");
    return ctrs;
}

uint64_t fuse_merkle_passes(const std::vector<MerkleArgs> &passes, MerkleArgs &out)
{
    if (passes.size() > (size_t)kMerkleMaxPasses) invalid("internal: Merkle pass plan");
    return fuse_merkle_passes(passes.data(), (uint32_t)passes.size(), out);
}

void launch_merkle_pass(hipStream_t stream, int hash_type, const MerkleArgs *dev_list,
                        uint32_t n, const MerkleArgs &one, uint64_t blocks, uint32_t tile_log_max, uint64_t chunk,
                        const char *name)
{
    if (blocks == 0) return;
    if (blocks > 0x7FFFFFFFull) invalid("tree too large for one launch");
    if (tile_log_max < (uint32_t)kMerkleMinTileLog || tile_log_max > (uint32_t)kMerkleMaxTileLog)
        invalid("Merkle tile size out of range");
    ProfScope ps(name, stream);
    const uint64_t step = (chunk && n > 0) ? chunk : blocks;
    for (uint64_t b0 = 0; b0 < blocks; b0 += step) {
        const uint64_t nb = std::min(step, blocks - b0);
        switch (hash_type) {
        case kPoseidon2: launch_merkle_hash<kPoseidon2>(stream, dev_list, n, one, nb, tile_log_max, (uint32_t)b0); break;
        case kKeccak: launch_merkle_hash<kKeccak>(stream, dev_list, n, one, nb, tile_log_max, (uint32_t)b0); break;
        case kMonolith: launch_merkle_hash<kMonolith>(stream, dev_list, n, one, nb, tile_log_max, (uint32_t)b0); break;
        case kPoseidonBN128:
            launch_merkle_hash<kPoseidonBN128>(stream, dev_list, n, one, nb, tile_log_max, (uint32_t)b0);
            break;
        default: launch_merkle_hash<kPoseidon>(stream, dev_list, n, one, nb, tile_log_max, (uint32_t)b0); break;
        }
        ZKX_HIP(hipGetLastError());
    }
}

MerkleArgs merkle_level_args(const MerkleArgs &leaf, uint32_t lg_w)
{
    MerkleArgs a{};
    a.dig = leaf.dig;
    a.cap = leaf.cap;
    a.sdl = leaf.sdl;
    a.lg_w = lg_w;
    a.count = (leaf.count >> leaf.lg_w) << lg_w;
    return a;
}

void launch_merkle_level(hipStream_t stream, int hash_type, const MerkleArgs *dev_list, uint32_t n, uint64_t blocks,
                         uint64_t chunk, const MerkleArgs &one)
{
    if (blocks == 0) return;
    if (blocks > 0x7FFFFFFFull) invalid("tree level too large for one launch");
    ProfScope ps("merkle_levels", stream);
    const uint64_t step = chunk ? chunk : blocks;
    for (uint64_t b0 = 0; b0 < blocks; b0 += step) {
        const uint64_t nb = std::min(step, blocks - b0);
        switch (hash_type) {
        case kPoseidon2: launch_merkle_level_hash<kPoseidon2>(stream, dev_list, n, one, nb, (uint32_t)b0); break;
        case kKeccak: launch_merkle_level_hash<kKeccak>(stream, dev_list, n, one, nb, (uint32_t)b0); break;
        case kMonolith: launch_merkle_level_hash<kMonolith>(stream, dev_list, n, one, nb, (uint32_t)b0); break;
        case kPoseidonBN128:
            launch_merkle_level_hash<kPoseidonBN128>(stream, dev_list, n, one, nb, (uint32_t)b0);
            break;
        default: launch_merkle_level_hash<kPoseidon>(stream, dev_list, n, one, nb, (uint32_t)b0); break;
        }
        ZKX_HIP(hipGetLastError());
    }
}

void launch_merkle_narrow(hipStream_t stream, int hash_type, const MerkleArgs *dev_list, uint32_t n,
                          const MerkleArgs &one, uint64_t blocks, const char *name, uint64_t chunk)
{
    if (blocks == 0) return;
    if (blocks > 0x7FFFFFFFull) invalid("tree too large for one launch");
    ProfScope ps(name, stream);
    const uint64_t step = (chunk && n > 0) ? chunk : blocks;
    for (uint64_t b0 = 0; b0 < blocks; b0 += step) {
        const uint64_t nb = std::min(step, blocks - b0);
        if (hash_type == kPoseidon2)
            launch_merkle_narrow_hash<kPoseidon2>(stream, dev_list, n, one, nb, (uint32_t)b0);
        else launch_merkle_narrow_hash<kPoseidon>(stream, dev_list, n, one, nb, (uint32_t)b0);
        ZKX_HIP(hipGetLastError());
    }
}

namespace {

uint32_t *device_counters(Device &d, uint64_t n) { return d.merkle_counters(n); }

MerkleArgs *device_descriptor(Device &d, const MerkleArgs &f)
{
    MerkleArgs *dj = d.merkle_descriptor();
    ZKX_HIP(hipMemcpyAsync(dj, &f, sizeof(f), hipMemcpyHostToDevice, d.stream));
    return dj;
}

// The tree, or what lies above the level of width 2^*written per subtree, in
// one launch.
void build_narrow(Device &d, const MerkleSpec &s, const uint32_t *written, const MerkleScratch &scratch)
{
    MerkleArgs f;
    const uint64_t nctr = plan_merkle_narrow(s, written, f);
    if (nctr) f.ctr = scratch.counters(d, nctr);
    if (has_tile_top(s.hash_type)) {
        const MerkleArgs *dj = scratch.descriptor(d, f);
        launch_merkle_pass(d.stream, (int)s.hash_type, dj, 1, MerkleArgs{}, f.count >> f.tile_log, kMerkleMinTileLog, 0,
                           "merkle_levels");
        return;
    }
    launch_merkle_narrow(d.stream, (int)s.hash_type, nullptr, 0, f, f.count >> f.tile_log,
                         f.leaves ? "merkle_narrow" : "merkle_levels");
}

}  // namespace

MerkleScratch device_merkle_scratch() { return MerkleScratch{device_counters, device_descriptor}; }

void merkle_build(Device &d, const MerkleSpec &s, const MerkleScratch &scratch)
{
    check_merkle(s);
    const Tuning tun = d.cabi_merkle_tuning(s.num_leaves, s.hash_type);
    const uint32_t tl = tun.merkle_tile_log;
    MerkleSpec sv = s;
    sv.leaf_valu = tun.merkle_valu;
    MerkleArgs passes[kMerkleMaxPasses];
    const uint32_t np = plan_merkle(sv, passes, tl);
    const uint64_t apart_from = d.lone_level_leaves.load();
    if (!tun.by_caller && lone_tree_narrow(s.num_leaves, s.hash_type, apart_from)) {
        build_narrow(d, s, nullptr, scratch);
        return;
    }
    if (s.num_caps < s.num_leaves && lone_tree_levels_apart(s.num_leaves, s.hash_type, apart_from)) {
        // a large tree: the leaf digests in one launch, then one launch per
        // level (k_merkle_level), each level's descriptor passed by value
        MerkleArgs leaf = passes[0];
        leaf.leaves_only = 1;
        launch_merkle_pass(d.stream, (int)s.hash_type, nullptr, 0, leaf, leaf.count >> leaf.tile_log, tl);
        for (uint32_t w = leaf.lg_w; w-- > 0;) {
            if ((has_narrow_kernel(s.hash_type) || has_tile_top(s.hash_type)) && s.num_caps << (w + 1) <= kNarrowNodes) {
                const uint32_t written = w + 1;
                build_narrow(d, s, &written, scratch);
                break;
            }
            const MerkleArgs lv = merkle_level_args(leaf, w);
            launch_merkle_level(d.stream, (int)s.hash_type, nullptr, 0,
                                (lv.count + kMerkleLevelLanes - 1) / kMerkleLevelLanes, 0, lv);
        }
        return;
    }
    MerkleArgs f;
    const uint64_t nctr = fuse_merkle_passes(passes, np, f);
    f.tile_begin = 0;
    if (!nctr) {
        launch_merkle_pass(d.stream, (int)s.hash_type, nullptr, 0, f, f.count >> f.tile_log, tl);
        return;
    }
    // fused upper passes read their fields from a descriptor in device memory
    f.ctr = scratch.counters(d, nctr);
    const MerkleArgs *dj = scratch.descriptor(d, f);
    launch_merkle_pass(d.stream, (int)s.hash_type, dj, 1, MerkleArgs{}, f.count >> f.tile_log, tl);
}

}  // namespace zkx
