// Merkle kernels hashing with Poseidon2 (hash type of merkle/merkle.h).
#include "merkle_launch_impl.h"

namespace zkx {

template void launch_merkle_hash<kPoseidon2>(hipStream_t, const MerkleArgs *, uint32_t, const MerkleArgs &, uint64_t,
                                     uint32_t, uint32_t);
template void launch_merkle_level_hash<kPoseidon2>(hipStream_t, const MerkleArgs *, uint32_t, const MerkleArgs &,
                                         uint64_t, uint32_t);
template void launch_merkle_narrow_hash<kPoseidon2>(hipStream_t, const MerkleArgs *, uint32_t, const MerkleArgs &, uint64_t,
                                         uint32_t);

}  // namespace zkx
