// Instantiates the FP32-shifted D2Q9 kernels for the E8 stencil.
#include "sc_impl.h"

const SimOps* get_ops_d2q9_e8_f32(int coll) {
  return idmx::ops_for_f32<D2Q9, D2E8>(coll);
}
