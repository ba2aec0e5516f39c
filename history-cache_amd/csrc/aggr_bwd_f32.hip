// The backward aggregation's kernels for a gradient of float rows.
#define BWD_INSTANTIATE
#include "aggr_bwd_rows.h"

int bwd_dispatch_f32(BwdArgs &a, bool masked, hipStream_t st) { return bwd_dispatch<float>(a, masked, st); }
