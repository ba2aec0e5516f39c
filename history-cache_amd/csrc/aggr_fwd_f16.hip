// The forward aggregation's kernels for __half rows.
#define FWD_INSTANTIATE
#include "aggr_fwd_rows.h"

int fwd_dispatch_f16(FwdArgs &a, bool src_mode, int n_head, hipStream_t st) {
  return dispatch<__half>(a, src_mode, n_head, st);
}
