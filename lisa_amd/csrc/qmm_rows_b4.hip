// Instantiations of the few-rows matmul (the kernel is in qmm_rows.h).
#include "qmm_rows.h"

namespace lisaq {

template <>
qmm_fn qmm_rows_get<4, kCtBf16>(int gs, int MT, int* lds) {
  return qmm_rows_get_impl<4, kCtBf16>(gs, MT, lds);
}

}  // namespace lisaq
