// Launches of the one-launch transforms (ntt_columns.h).
#include "ntt_columns.h"

#include "ntt.h"

namespace zkx {

namespace {

template <int LT, int LE, int L>
void launch(hipStream_t s, const NttPass *list, uint32_t n, const NttPass &one, const ColumnPost &post, bool inverse,
            uint64_t first, uint64_t end)
{
    const dim3 grid((uint32_t)(end - first)), block(1 << (LT - LE));
    if (inverse) hipLaunchKernelGGL((k_ntt_columns<LT, LE, L, true>), grid, block, 0, s, list, n, one, post, first);
    else hipLaunchKernelGGL((k_ntt_columns<LT, LE, L, false>), grid, block, 0, s, list, n, one, post, first);
}

}  // namespace

void launch_columns(hipStream_t s, uint32_t L, uint32_t tile_log, const NttPass *list, uint32_t n, const NttPass &one,
                    const ColumnPost &post, bool inverse, uint64_t first, uint64_t end)
{
#define ZKX_COLUMNS(LT, LE, LL) \
    case LT * 100 + LL: return launch<LT, LE, LL>(s, list, n, one, post, inverse, first, end)
    switch (tile_log * 100 + L) {
        ZKX_COLUMNS(12, 2, 1);
        ZKX_COLUMNS(12, 2, 2);
        ZKX_COLUMNS(12, 2, 3);
        ZKX_COLUMNS(12, 2, 4);
        ZKX_COLUMNS(12, 2, 5);
        ZKX_COLUMNS(12, 2, 6);
        ZKX_COLUMNS(12, 2, 7);
        ZKX_COLUMNS(12, 2, 8);
        ZKX_COLUMNS(12, 2, 9);
        ZKX_COLUMNS(12, 2, 10);
        ZKX_COLUMNS(12, 2, 11);
        ZKX_COLUMNS(12, 2, 12);
        ZKX_COLUMNS(13, 3, 10);
        ZKX_COLUMNS(13, 3, 11);
        ZKX_COLUMNS(13, 3, 12);
        ZKX_COLUMNS(13, 3, 13);
        ZKX_COLUMNS(14, 4, 11);
        ZKX_COLUMNS(14, 4, 12);
        ZKX_COLUMNS(14, 4, 13);
        ZKX_COLUMNS(14, 4, 14);
    }
#undef ZKX_COLUMNS
    invalid("internal: no one-launch transform of this size");
}

}  // namespace zkx
