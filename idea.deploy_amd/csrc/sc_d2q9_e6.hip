// Instantiates the FP64 D2Q9 kernels for the E6 stencil (compiled without
// floating-point contraction).
#include "sc_impl.h"

const SimOps* get_ops_d2q9_e6_f64(int coll) {
  return idmx::ops_for_f64<D2Q9, D2E6>(coll);
}
