// The backward aggregation's kernels for a gradient of __half rows.
#define BWD_INSTANTIATE
#include "aggr_bwd_rows.h"

int bwd_dispatch_f16(BwdArgs &a, bool masked, hipStream_t st) { return bwd_dispatch<__half>(a, masked, st); }
