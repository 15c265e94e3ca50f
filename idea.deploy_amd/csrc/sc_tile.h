// sc_tile.h -- four time steps of a small D2Q9 lattice (E4 force) in one
// launch.
//
// What bounds a small lattice is latency: a step of 128^2 sites moves 2.4 MB
// that stay in L2 and is over in 5.2 us, most of it launch, two memory
// latencies and a barrier. A block here loads a B x B tile with the ring of
// sites that KS steps reach, takes the steps in LDS on a region that shrinks
// by two sites per side and step, and pushes the result: one launch and one
// round trip to memory per KS steps, paid for with redundant collisions on
// the ring (KS = 4: 3.4 times the sites of an 8 x 8 tile, 2.0 of a 16 x 16
// one), which an otherwise idle chip has room for. Measured per step against
// the register step, one launch each: 128^2 1.92 us (5.10), 256^2 2.53 (6.06),
// 384^2 6.6 (8.6), 512^2 9.5 (11.0).
//
// One site per thread: thread t is site (t mod w, t / w) of the stage's
// region of w x w sites, where psi is needed (PW); it collides there unless
// it lies on the region's rim.
#pragma once
#include <type_traits>

#include "sc_kernels.h"

namespace idmx {

template <int B, int KS>
struct TileShape {
  static constexpr int PW(int s) { return B + 4 * (KS - 1 - s) + 2; }  // psi of stage s
  static constexpr int CW(int s) { return PW(s) - 2; }                 // collisions
  static constexpr int NT = (PW(0) * PW(0) + 63) / 64 * 64;
  // f* of even and odd stages (that of the last one goes to memory)
  static constexpr int F0 = CW(0) * CW(0), F1 = KS > 2 ? CW(1) * CW(1) : 1;
};

template <class T, bool SHIFT, int COLL, int B, int KS, bool WF>
__global__ void __launch_bounds__((TileShape<B, KS>::NT))
k_tile2d(const T* __restrict__ pop, T* __restrict__ pop_swap, Geom geo, Phys<T> P, int ntx,
         int ntiles, double* __restrict__ n_out, double* __restrict__ psi_out,
         double* __restrict__ u_out) {
  using S = D2Q9;
  using ES = D2E4;
  using SH = TileShape<B, KS>;
  constexpr int Q = S::Q, NB = NBasis<2>::value;
  constexpr int NTAB = COLL == 2 ? Q : COLL == 1 ? Q * Q + 2 * NB * Q : 1;
  __shared__ T fa[Q][SH::F0], fb[Q][SH::F1];
  __shared__ T pa[SH::PW(0) * SH::PW(0)], pb[SH::PW(1) * SH::PW(1)];
  __shared__ T tab[NTAB];
  const int per = gridDim.x >> 3;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (tile >= ntiles) return;
  const int x0 = tile % ntx * B, y0 = tile / ntx * B;
  const int tid = threadIdx.x;
  Phys<T> PL = P;
  if constexpr (COLL == 1 || COLL == 2) {
    for (int i = tid; i < NTAB; i += SH::NT) tab[i] = P.mrtA[i];
    PL.mrtA = tab;
    PL.mrtB = COLL == 1 ? tab + Q * Q : nullptr;
    PL.mrtG = COLL == 1 ? tab + Q * Q + NB * Q : nullptr;
  }
  auto stage = [&](auto sc, const T* fin, int fin_n, T* fout, int fout_n, T* psi) {
    constexpr int s = sc.value, PW = SH::PW(s), CW = SH::CW(s);
    constexpr int IW = s > 0 ? SH::CW(s - 1) : 1;  // width of the region fin covers
    const bool in = tid < PW * PW;
    const int px = tid % PW, py = tid / PW;
    T f[Q], dn = T(0);
    if (in) {
      if constexpr (s == 0) {
        const int D = 2 * KS - 1;
        const int x = ((x0 - D + px) % geo.L0 + geo.L0) % geo.L0;
        const int y = ((y0 - D + py) % geo.L1 + geo.L1) % geo.L1;
        const int64_t g = (int64_t)y * geo.L0 + x;
#pragma unroll
        for (int q = 0; q < Q; q++) f[q] = pop_ld(pop, q, geo.V, g);
      } else {
        // f streamed from the previous stage's f*: its region reaches one
        // site further on every side
#pragma unroll
        for (int q = 0; q < Q; q++)
          f[q] = fin[q * fin_n + (py + 1 - S::cy[q]) * IW + px + 1 - S::cx[q]];
      }
      dn = f[0];
#pragma unroll
      for (int q = 1; q < Q; q++) dn += f[q];
      psi[tid] = psi_of(P.psi_kind, SHIFT ? P.rho0 + dn : dn);
    }
    __syncthreads();
    if (in && px > 0 && px < PW - 1 && py > 0 && py < PW - 1) {
      T gx, gy, gz, fo[Q], u[3];
      iso_grad<ES>([&](int e) { return psi[tid + ES::ey[e] * PW + ES::ex[e]]; }, gx, gy, gz);
      const T lpsi = psi[tid];
      collide<S, T, SHIFT, COLL>(f, dn, gx, gy, T(0), lpsi, PL, fo, u);
      if constexpr (s < KS - 1) {
        const int c = (py - 1) * CW + px - 1;
#pragma unroll
        for (int q = 0; q < Q; q++) fout[q * fout_n + c] = fo[q];
      } else {
        const int x = x0 + px - 1, y = y0 + py - 1;
        if (x < geo.L0 && y < geo.L1) {
          push_store<S, T>(pop_swap, geo, x, y, 0, fo);
          if (WF) {
            const int64_t g = (int64_t)x + (int64_t)geo.L0 * y;
            n_out[g] = (double)(SHIFT ? P.rho0 + dn : dn);
            psi_out[g] = (double)lpsi;
            u_out[g] = (double)u[0];
            u_out[g + geo.V] = (double)u[1];
          }
        }
      }
    }
    if constexpr (s < KS - 1) __syncthreads();
  };
  static_assert(KS == 4, "stages are written out");
  stage(std::integral_constant<int, 0>{}, nullptr, 0, fa[0], SH::F0, pa);
  stage(std::integral_constant<int, 1>{}, fa[0], SH::F0, fb[0], SH::F1, pb);
  stage(std::integral_constant<int, 2>{}, fb[0], SH::F1, fa[0], SH::F0, pa);
  stage(std::integral_constant<int, 3>{}, fa[0], SH::F0, nullptr, 0, pb);
}

}  // namespace idmx
