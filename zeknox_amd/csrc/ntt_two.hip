// Launches of the two-launch transforms (ntt_two.h).
#include "ntt_two.h"

#include "ntt.h"

namespace zkx {

namespace {

template <int M>
void first(hipStream_t s, const NttPass &a, uint32_t tiles)
{
    if (a.inverse) hipLaunchKernelGGL((k_ntt_first<M, true>), dim3(tiles), dim3(kTwoLanes), 0, s, a);
    else hipLaunchKernelGGL((k_ntt_first<M, false>), dim3(tiles), dim3(kTwoLanes), 0, s, a);
}

template <int M>
void second(hipStream_t s, const NttPass &a, const ColumnPost &post, uint32_t tiles)
{
    if (a.inverse) hipLaunchKernelGGL((k_ntt_second<M, true>), dim3(tiles), dim3(kTwoLanes), 0, s, a, post);
    else hipLaunchKernelGGL((k_ntt_second<M, false>), dim3(tiles), dim3(kTwoLanes), 0, s, a, post);
}

}  // namespace

void launch_two_first(hipStream_t s, const NttPass &a)
{
    const uint32_t tiles = (uint32_t)(a.total >> kTwoTile);
    switch (a.m) {
    case 8: return first<8>(s, a, tiles);
    case 9: return first<9>(s, a, tiles);
    case 10: return first<10>(s, a, tiles);
    }
    invalid("internal: no two-launch transform of this size");
}

void launch_two_second(hipStream_t s, const NttPass &a, const ColumnPost &post)
{
    const uint32_t tiles = (uint32_t)(a.total >> kTwoTile);
    switch (a.m) {
    case 7: return second<7>(s, a, post, tiles);
    case 8: return second<8>(s, a, post, tiles);
    case 9: return second<9>(s, a, post, tiles);
    case 10: return second<10>(s, a, post, tiles);
    }
    invalid("internal: no two-launch transform of this size");
}

}  // namespace zkx
