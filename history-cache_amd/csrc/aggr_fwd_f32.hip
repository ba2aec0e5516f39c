// The forward aggregation's kernels for float rows.
#define FWD_INSTANTIATE
#include "aggr_fwd_rows.h"

int fwd_dispatch_f32(FwdArgs &a, bool src_mode, int n_head, hipStream_t st) {
  return dispatch<float>(a, src_mode, n_head, st);
}
