// Instantiations of the qmm kernel for bf16 and 8-bit codes, with and without
// split-K partial output (the kernel is in qmm_kernel.h).
#include "qmm_kernel.h"

namespace lisaq {

template <>
qmm_fn qmm_get<8, false, kCtBf16>(int gs, int MT, bool odd, int* lds) {
  return qmm_get_impl<8, false, kCtBf16>(gs, MT, odd, lds);
}

template <>
qmm_fn qmm_get<8, true, kCtBf16>(int gs, int MT, bool odd, int* lds) {
  return qmm_get_impl<8, true, kCtBf16>(gs, MT, odd, lds);
}

}  // namespace lisaq
