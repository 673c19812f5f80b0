// The wide kernels of FP32 products with a materialised operator whose unit stride runs
// along the output's rows.
#include "rbx_wide.hh"

RBX_WIDE_INSTANCES(float, WIDE_MEM, true)
