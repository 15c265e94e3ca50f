// Instantiates the FP32-shifted D2Q9 kernels for the E6 stencil.
#include "sc_impl.h"

const SimOps* get_ops_d2q9_e6_f32(int coll) {
  return idmx::ops_for_f32<D2Q9, D2E6>(coll);
}
