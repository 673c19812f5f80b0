// The wide kernels of FP32 products with a materialised operator whose unit stride runs
// along the contraction.
#include "rbx_wide.hh"

RBX_WIDE_INSTANCES(float, WIDE_PRE, false)
