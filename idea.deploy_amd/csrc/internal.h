// internal.h -- context/simulation objects shared by the translation units of
// libidmx.so (not part of the C ABI).
#pragma once
#include <hip/hip_runtime.h>

#include <string>
#include <vector>

#include "../../include/idmx.h"
#include "sc_kernels.h"

namespace idmx {

void set_error(const std::string& msg);
int hip_fail(hipError_t e, const char* what);

#define IDMX_HIP(call)                                        \
  do {                                                        \
    hipError_t e_ = (call);                                   \
    if (e_ != hipSuccess) return ::idmx::hip_fail(e_, #call); \
  } while (0)

}  // namespace idmx

struct idmx_ctx_s {
  int device = 0;
  hipStream_t stream = nullptr;
  double* partials = nullptr;      // device scratch for reductions
  size_t partials_cap = 0;         // in doubles
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  float* nn_part = nullptr;        // per-block weight gradients of the network
  size_t nn_part_cap = 0;          // in floats; grown on demand, freed with the context
};

struct SimOps;

// Sites below which a 3D simulation that was given no launch takes its steps
// without a march (k_tile3d): 24^3 MRT 7.6 us per step against 13.1, 48 x 44 x
// 40 11.6 against 14.1 (E8: 16.5 against 19.5), 60 x 50 x 48 BGK 19.3 against
// 21.4, 64^3 25.9 against 23.6; in FP32 48 x 44 x 40 8.4 against 10.4, 50^3
// 13.7 against 12.7.
constexpr int64_t kTile3Sites = 150000, kTile3Sites32 = 100000;

// March length of a 3D step of which two blocks share a CU: the launch runs in
// rounds of 512 blocks of h + 2R planes each, and the least total wins (half a
// plane for a block's start). `tiles` per plane, Lm planes; *cost: the total.
inline int march_planes(int64_t tiles, int Lm, int R, double* cost = nullptr) {
  double least = 1e300;
  int best = Lm;
  for (int nseg = 1; nseg <= std::min(Lm, 4096); nseg++) {
    const int h = (Lm + nseg - 1) / nseg;
    const int64_t rounds = (tiles * ((Lm + h - 1) / h) + 511) / 512;
    const double c = (double)rounds * (h + 2 * R + 0.5);
    if (c < least) least = c, best = h;
  }
  if (cost) *cost = least;
  return best;
}

struct idmx_sc_s {
  idmx_ctx_s* ctx = nullptr;
  idmx_sc_desc desc{};
  int D = 0, Q = 0;
  idmx::Geom geo{};
  size_t pop_elem = 8;       // bytes per population value
  void* mrt_dev = nullptr;   // MRT tables in the working precision
  idmx::PsiProg* psi_prog_dev = nullptr;  // psi_kind 3: the compiled psi_code
  uint32_t* wflag_host = nullptr;  // pinned: set where a wall flag is neither 0 nor 1
  uint64_t* wmask_dev = nullptr;  // V wall masks of the fused step with walls
  double last_ms = 0;
  const SimOps* ops = nullptr;
  // fused launch shape (chosen at create time, autotuner may override)
  int tx = 0, ty = 0, H = 0, hist = 1;
  // the launch chosen at creation (tx, ty, H, hist), and whether it is in
  // force: it includes a step and a march length that the four do not name
  int first_launch[4] = {0, 0, 0, 0};
  bool auto_launch = true;
  int xsh = 0;  // variant 10: the running step's x-shifted storage flags
  int coll = 0;  // 0 BGK, 1 dense MRT, 2 diagonal MRT, 3 BGK with Shan-Chen forcing,
                 // 4 BGK followed by the isotropy filter
  const uint8_t* walls = nullptr;  // device flags, 1 fluid / 0 solid (borrowed)
  // per-step timing of idmx_sc_run_profiled: 2 events per step + 1, reused
  std::vector<hipEvent_t> prof_ev;
  float* prof_ms = nullptr;  // 2 * nsteps host floats while a profiled run is active
  double bforce[3] = {0.0, 0.0, 0.0};  // body force added to the Shan-Chen force
};

// Per-(velocity set, E-stencil, precision, collision) entry points.
struct SimOps {
  int (*run)(idmx_sc_s*, void** pop, void** swap, double* n, double* psi,
             double* u, int nsteps, int flags);
  int (*density_psi)(idmx_sc_s*, double* n, double* psi, const void* pop);
  int (*fcs)(idmx_sc_s*, void* swap, const void* pop, const double* n,
             const double* psi, double* u);
  int (*moments)(idmx_sc_s*, const void* pop, double* n, double* psi, double* u);
  int (*density_velocity)(idmx_sc_s*, const void* pop, double* n, double* u);
  int (*init_pop)(idmx_sc_s*, void* pop, const double* n, const double* u);
  int (*mass_mom)(idmx_sc_s*, const void* pop, double* mass, double* mom);
  int (*to_f64)(idmx_sc_s*, const void* pop, double* dst);
  int (*from_f64)(idmx_sc_s*, void* pop, const double* src);
  int (*launch_ok)(int tx, int ty, int variant);
  int (*init_pop_tab)(idmx_sc_s*, void* pop, const double* n, const double* u,
                      const double* coeffs);
};

// One unit per velocity set, stencil and precision: a simulation's first launch
// loads the whole unit that the kernel is in.
const SimOps* get_ops_d2q9_e4_f64(int coll);
const SimOps* get_ops_d2q9_e4_f32(int coll);
const SimOps* get_ops_d2q9_e6_f64(int coll);
const SimOps* get_ops_d2q9_e6_f32(int coll);
const SimOps* get_ops_d2q9_e8_f64(int coll);
const SimOps* get_ops_d2q9_e8_f32(int coll);
const SimOps* get_ops_d3q19_e4_f64(int coll);
const SimOps* get_ops_d3q19_e4_f32(int coll);
const SimOps* get_ops_d3q19_e6_f64(int coll);
const SimOps* get_ops_d3q19_e6_f32(int coll);
const SimOps* get_ops_d3q19_e8_f64(int coll);
const SimOps* get_ops_d3q19_e8_f32(int coll);
