// Instantiations of the qmm kernel for 2-bit codes, split-K partial output
// (one of four translation units compiled in parallel; the kernel is in qmm_kernel.h).
#include "qmm_kernel.h"

namespace lisaq {

template <>
qmm_fn qmm_get<2, true>(int gs, int MT, bool odd, int* lds) {
  return qmm_get_impl<2, true>(gs, MT, odd, lds);
}

}  // namespace lisaq
