// The wide kernels of FP64 products with a Gaussian operator whose counters run
// along the output's rows.
#include "rbx_wide.hh"

RBX_WIDE_INSTANCES(double, WIDE_GAUSS, true)
