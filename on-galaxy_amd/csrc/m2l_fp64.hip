// ============================================================================
// m2l_fp64.hip -- the FP64 M2L's entry point (kernel: m2l_fp64_kernel.h,
// compiled per order by m2l_fp64_order.hip).
// ============================================================================
#include <stdexcept>

#include "afmm_internal.h"

namespace afmm {

template <int P>
void m2l_fp64_launch(hipStream_t s, const M2LArgs& a);

void m2l_fp64(hipStream_t s, int p, const M2LArgs& a) {
    switch (p) {
#define AFMM_CASE(PP) \
    case PP: m2l_fp64_launch<PP>(s, a); return;
        AFMM_CASE(1) AFMM_CASE(2) AFMM_CASE(3) AFMM_CASE(4) AFMM_CASE(5) AFMM_CASE(6)
        AFMM_CASE(7) AFMM_CASE(8) AFMM_CASE(9) AFMM_CASE(10) AFMM_CASE(11) AFMM_CASE(12)
        AFMM_CASE(13) AFMM_CASE(14) AFMM_CASE(15) AFMM_CASE(16)
#undef AFMM_CASE
    }
    throw std::runtime_error("unsupported expansion order");
}

}  // namespace afmm
