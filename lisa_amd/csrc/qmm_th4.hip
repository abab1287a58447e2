// Instantiations of the qmm kernel for f16 and 4-bit codes, with and without
// split-K partial output (the kernel is in qmm_kernel.h).
#include "qmm_kernel.h"

namespace lisaq {

template <>
qmm_fn qmm_get<4, false, kCtF16>(int gs, int MT, bool odd, int* lds) {
  return qmm_get_impl<4, false, kCtF16>(gs, MT, odd, lds);
}

template <>
qmm_fn qmm_get<4, true, kCtF16>(int gs, int MT, bool odd, int* lds) {
  return qmm_get_impl<4, true, kCtF16>(gs, MT, odd, lds);
}

}  // namespace lisaq
