// The forward aggregation's kernels for __hip_bfloat16 rows.
#define FWD_INSTANTIATE
#include "aggr_fwd_rows.h"

int fwd_dispatch_bf16(FwdArgs &a, bool src_mode, int n_head, hipStream_t st) {
  return dispatch<__hip_bfloat16>(a, src_mode, n_head, st);
}
