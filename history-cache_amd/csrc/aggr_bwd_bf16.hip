// The backward aggregation's kernels for a gradient of __hip_bfloat16 rows.
#define BWD_INSTANTIATE
#include "aggr_bwd_rows.h"

int bwd_dispatch_bf16(BwdArgs &a, bool masked, hipStream_t st) { return bwd_dispatch<__hip_bfloat16>(a, masked, st); }
