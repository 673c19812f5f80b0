// The wide kernels of FP64 products with a materialised operator whose unit stride runs
// along the contraction.
#include "rbx_wide.hh"

RBX_WIDE_INSTANCES(double, WIDE_PRE, false)
