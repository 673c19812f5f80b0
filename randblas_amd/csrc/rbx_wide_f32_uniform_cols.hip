// The wide kernels of FP32 products with a uniform operator whose counters run
// along the contraction.
#include "rbx_wide.hh"

RBX_WIDE_INSTANCES(float, WIDE_UNIFORM, false)
