// Instantiates the FP64 D2Q9 kernels for the E8 stencil (compiled without
// floating-point contraction).
#include "sc_impl.h"

const SimOps* get_ops_d2q9_e8_f64(int coll) {
  return idmx::ops_for_f64<D2Q9, D2E8>(coll);
}
