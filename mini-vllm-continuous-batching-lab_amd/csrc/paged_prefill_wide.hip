// Prefill attention with 256 packed query rows per work group (the 16-bit
// types; mv_prefill16.h): eight row waves and no key sets. A pass over the keys
// serves twice the rows of a 128-row group: half the copies into LDS and no set
// merge, but half the groups, each with its keys in one chain. Measured
// against 128 rows (units of 128 rows; 256 CUs): where whole rounds over the
// CUs come out alike it wins, 14 / 2 heads x 64 bf16, 16 x (1536 + 512) (928
// units) 82.5 -> 75.4 us; 28 / 4 x 128, 7 x (1536 + 504) (784) 131 -> 108, one
// 8192-token prompt (1824) 473 -> 434; where they do not it loses, 4 x (1536 +
// 512) at 14 / 2 x 64 (232) 26.6 -> 53.6, 5120 tokens over 1536 at 8 / 8 x 64
// fp16 (320) 68 -> 113, a 4608-token prompt at 14 / 2 x 64 (512) 56 -> 81.
#include "mv_prefill16.h"

namespace mv {
namespace {

template <int DTYPE, int D, typename BT>
__global__ __launch_bounds__(512) void paged_prefill_wide_kernel(PrefillArgs a) {
  prefill16<Prefill16Traits<DTYPE, D, 8, 1>, BT>(a);
}

template <int DTYPE, int D>
void launch(const PrefillArgs& a, int groups, bool bt_i64, hipStream_t s) {
  if (bt_i64) paged_prefill_wide_kernel<DTYPE, D, int64_t><<<groups, 512, 0, s>>>(a);
  else paged_prefill_wide_kernel<DTYPE, D, int32_t><<<groups, 512, 0, s>>>(a);
}

}  // namespace

int launch_prefill_wide(const PrefillArgs& a, int head_dim, int dtype, int groups, bool bt_i64, hipStream_t s) {
  if (dtype == MV_DTYPE_F16) {
    if (head_dim == 64) launch<MV_DTYPE_F16, 64>(a, groups, bt_i64, s);
    else launch<MV_DTYPE_F16, 128>(a, groups, bt_i64, s);
  } else {
    if (head_dim == 64) launch<MV_DTYPE_BF16, 64>(a, groups, bt_i64, s);
    else launch<MV_DTYPE_BF16, 128>(a, groups, bt_i64, s);
  }
  return check_launch("mv_paged_prefill (wide)");
}

}  // namespace mv
