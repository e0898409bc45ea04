// Host-side NTT / LDE / transpose drivers (device pointers, enqueued on the
// device's stream; the caller synchronises).
#pragma once
#include <vector>

#include "ntt_types.h"
#include "runtime.h"
#include "tuning.h"

namespace zkx {

// LDE of `cols` columns of 2^lg_n coefficients into `out` (cols x 2^(lg_n+rate)),
// each output column in bit-reversed order (DIF order, no reversal pass).
void lde_bitrev(Device &d, uint64_t *out, const uint64_t *in, uint32_t lg_n, uint32_t rate, uint32_t cols,
                bool inverse, bool with_coset);
// Resident LDE factor table F[b*n + i] = (g * w_N^{bitrev_r(b)})^i (g = 1
// without coset; w^-1 for the inverse), built on first use.
const uint64_t *lde_factor_table(Device &d, uint32_t lg_n, uint32_t rate, bool inverse, bool with_coset);
// compute_batched_lde semantics: natural-order output.
void lde(Device &d, uint64_t *out, const uint64_t *in, uint32_t lg_n, uint32_t rate, uint32_t cols,
         bool inverse, bool with_coset);
// compute_batched_ntt semantics: in place, natural order.
void ntt(Device &d, uint64_t *inout, uint32_t lg, uint32_t cols, bool inverse, bool with_coset);
// In-place bit reversal of each column with optional post-scaling.
void bitrev_columns(Device &d, uint64_t *buf, uint32_t lg, uint32_t cols, bool use_scale, uint64_t scale,
                    const uint64_t *coset);
// out[t * cols + b] = in[b * 2^lg + (rev ? bitrev(t) : t)].
void transpose_rev(Device &d, uint64_t *out, const uint64_t *in, uint32_t lg, uint32_t cols, bool rev);

// Pass descriptors of the DIF over nblk blocks of 2^L in buf (in launch
// order; each pass must finish before the next starts), cut into passes as
// `tun` says.  Returns the tile count of every pass.
// tw_lg: the device array of twiddle tables by log size, built up to L
// (Device::twiddle_tables_upto).
uint64_t plan_dif(std::vector<NttPass> &out, uint64_t *buf, uint64_t nblk, uint32_t L, uint32_t lg_tw,
                  const uint64_t *tw, const uint64_t *tw12, const uint64_t *const *tw_lg, bool inverse,
                  uint32_t mode0, const uint64_t *src, uint32_t rate, bool with_coset, const uint64_t *coset,
                  const Tuning &tun);

// Stage counts of the DIF passes over blocks of 2^L under `tun`, top
// stages first (the last pass contiguous).
std::vector<uint32_t> ntt_pass_sizes(uint32_t L, const Tuning &tun);
// The same for the forward LDE from coefficients (plan_dif with kSrcLde),
// which has one-launch blocks of 2^13 unless the caller set the schedule.
std::vector<uint32_t> lde_pass_sizes(uint32_t L, const Tuning &tun);

// Which register-round kernel a launch over these passes can use (each runs
// one tile per work-group): 0 none (k_ntt_tiles); 1 contiguous (every pass
// in place and a whole number of tiles; stages above 8 in registers);
// 2 + 4 * lde + (m - 1) strided single-round (every pass strided with the
// same m <= 4 stages and the same source, in place or LDE; registers only);
// 10 + 4 * lde + (m - 5) strided two-round (the same with 5 <= m <= 8, the
// first round in registers); kColumnKind + m whole blocks of 2^m <= 2^13 from
// coefficients, forward, every pass with the same m (ntt_columns.h).
constexpr int kColumnKind = 18;
int ntt_kernel_kind(const NttPass *host_list, size_t n);

// One launch over n pass descriptors in device memory (sorted by
// tile_begin), all contiguous (s_lo == 0) or all strided; `kernel_kind` as
// ntt_kernel_kind of the same list.  chunk > 0: launches over ranges of at
// most `chunk` tiles instead, in order (other streams' kernels can be
// dispatched between them).
void launch_ntt_list(hipStream_t stream, const NttPass *dev_list, uint32_t n, uint64_t blocks, bool contiguous,
                     int kernel_kind, const char *name, uint64_t chunk = 0);

// log2 words of the tile in which one launch does a whole transform of stages
// L into `cols` columns of 2^lg in natural order, 0 where passes and a bit
// reversal are used.  Rates above 3 have no kernel at 2^13 and 2^14.  A
// column of 2^14 takes a CU to itself, so few of them leave the chip to 31 us
// of passes that spread over it (inverse, one launch / passes, us: 2^14 x 20
// 37 / 34, x 101 39 / 54, x 400 71 / 98; 2^13 x 1 25 / 30, x 101 27 / 39,
// x 400 39 / 65; 2^12 x 1 20 / 27, x 400 27 / 44).
inline uint32_t column_tile_log(uint32_t L, uint32_t lg, uint32_t cols)
{
    if (L == 0 || L > lg) return 0;
    if (lg <= 12) return 12;
    if (lg > 14 || lg - L > 3) return 0;
    return lg == 13 || cols >= 48 ? lg : 0;
}
// That launch over the tiles [first, end) of the passes (device list, or
// `one` when n == 0): s_lo == 0, m == L, every mode.
void launch_columns(hipStream_t s, uint32_t L, uint32_t tile_log, const NttPass *list, uint32_t n, const NttPass &one,
                    const ColumnPost &post, bool inverse, uint64_t first, uint64_t end);

// The two launches of ntt_two.h over a.total words (whole columns): the top
// a.m stages from a.src into a.buf, and the low a.m stages from a.src into
// natural order in a.buf.
void launch_two_first(hipStream_t s, const NttPass &a);
void launch_two_second(hipStream_t s, const NttPass &a, const ColumnPost &post);

// table[i] = base^i, i < n.
void fill_powers(uint64_t *dst, uint64_t n, uint64_t base, hipStream_t s);
// `count` pseudo-random field elements from `seed` (LDE salt columns).
void fill_salt(uint64_t *dst, uint64_t count, uint64_t seed, hipStream_t s);

}  // namespace zkx
