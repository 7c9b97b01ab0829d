// ============================================================================
// m2l_fp64_order.hip -- the FP64 M2L of one expansion order, M2L_ORDER (the
// Makefile compiles this file once per order, side by side).
// ============================================================================
#include "m2l_fp64_kernel.h"

namespace afmm {
template void m2l_fp64_launch<M2L_ORDER>(hipStream_t, const M2LArgs&);
}  // namespace afmm
