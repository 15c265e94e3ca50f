// sc_pair.h -- two time steps of a D2Q9 lattice in one pass over the
// populations (the single-domain step on the x-shifted storage, 2D).
//
// What bounds it: a single step is bound by HBM (144 B per site and step in
// FP64); two steps per pass move 86 (4096^2 E8, measured), and the FP64 vector
// units and the latency of two waves per SIMD take over (vector units issuing
// in 54 % of the cycles, 4.6 TB/s). Measured per step on one MI355X, against
// the best single-step launch: 4096^2 E8 306 us (532), 4096^2 E4 291 us (520),
// 1000 x 613 Shan-Chen forcing 13.7 us (30), 1024^2 MRT 23 us (38.5), 4096^2
// FP32 161 us (270).
//
// Layout: a block of NT threads owns a strip of NT columns, of which the
// inner TXMAX or fewer are written, and marches along y; a thread keeps its
// column through both steps. Per iteration j:
//   phase 1  psi(0) of row j from the populations loaded in the previous
//            iteration (the load of row j + 1 is issued here, so it is in
//            flight during both collisions); f(1) of row j - R - 2 gathered
//            from the staged f*(0), its psi(1);
//   phase 2  the first step's collision of row j - R, f*(0) staged in LDS at
//            its target; the second step's collision of row j - 2R - 2, f*(1)
//            pushed to memory.
// Each phase reads what the other wrote, hence two barriers per iteration,
// and the two collisions of phase 2 are independent. Staging f*(0) by target
// keeps a population with c_qy = +1 for three rows, 0 for two, -1 for one:
// 16 rows of NT + 2 values instead of 27, so that E8 in FP64 needs 54 KB.
// Threads beyond the written columns compute values that only the threads up
// to HALO columns inwards read, and values nobody reads at the very edge
// (from LDS padding that is never written).
#pragma once
#include <type_traits>

#include "sc_kernels.h"

namespace idmx {

template <class ES, class T, int COLL, int NT, bool WALLS = false>
struct PairShape {
  static constexpr int R = ES::R;
  static constexpr int HALO = 2 * R + 1;  // columns (rows) of f(0) beyond the written ones
  static constexpr int TXMAX = NT - 2 * HALO;
  static constexpr int FX = NT + 2;       // row of a staged f*(0) population
  static constexpr int PX = NT + 2 * R;   // row of psi
  static constexpr int NS = 2 * R + 1;    // psi ring rows
  // rows kept of f*(0) by c_qy: +1 three, 0 two, -1 one (the rest population
  // stays in registers); with walls -1 two, since a population that bounces
  // back is staged one row above the pushed ones
  static constexpr int DOWN = WALLS ? 2 : 1;
  static constexpr int FROWS = 3 * 3 + 2 * 2 + 3 * DOWN;
  static constexpr int NB = NBasis<2>::value;
  static constexpr int Q = D2Q9::Q;
  static constexpr int NTAB = COLL == 2 ? Q : COLL == 1 ? Q * Q + 2 * NB * Q : 1;
};

// geo.L1 rows by H per block, txo columns written per block; xsh as in
// k_fused_dma (bit 0: reads the x-shifted storage, bit 1: writes it); WF: the
// second step also writes n, psi and u. Compiled for two waves per SIMD: at
// three the E4 step spills (4096^2, at an earlier state: 296 us instead of 286).
// WALLS: as in k_fused_dma, flags 0 and 1 only (with others the results are
// dropped by Impl::run); psi_out holds the psi of the solid sites, which
// stays, wmask the masks.
template <class ES, class T, bool SHIFT, int COLL, int NT, bool WF, bool WALLS = false>
__global__ void __launch_bounds__(NT, 2)
k_pair2d(const T* __restrict__ pop, T* __restrict__ pop_swap, Geom geo, Phys<T> P, int txo,
         int H, int ntx, int ntiles, int xsh, double* __restrict__ n_out,
         double* psi_out, double* __restrict__ u_out, const uint64_t* __restrict__ wmask = nullptr,
         T bx = T(0), T by = T(0)) {
  using S = D2Q9;
  using SH = PairShape<ES, T, COLL, NT, WALLS>;
  static_assert(!WALLS || (ES::R == 1 && sizeof(T) == 8 && !SHIFT));
  constexpr int Q = S::Q, R = ES::R, HALO = SH::HALO, NS = SH::NS;
  __shared__ T frow[SH::FROWS][SH::FX];
  __shared__ T ring0[NS][SH::PX], ring1[NS][SH::PX];
  __shared__ T tab[SH::NTAB];

  const int per = gridDim.x >> 3;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (tile >= ntiles) return;
  const int x0 = (tile % ntx) * txo, m0 = (tile / ntx) * H;
  const int Lm = geo.L1;
  const int Hs = min(H, Lm - m0);
  const int J = Hs + 2 * HALO + 1;
  const int tid = threadIdx.x;

  Phys<T> PL = P;
  if constexpr (COLL == 1 || COLL == 2) {
    for (int i = tid; i < SH::NTAB; i += NT) tab[i] = P.mrtA[i];
    PL.mrtA = tab;
    PL.mrtB = COLL == 1 ? tab + Q * Q : nullptr;
    PL.mrtG = COLL == 1 ? tab + Q * Q + SH::NB * Q : nullptr;
  }

  const int x = x0 - HALO + tid;
  const bool own = tid >= HALO && tid < HALO + txo && x < geo.L0;
  const int gx = ((x % geo.L0) + geo.L0) % geo.L0;
  const bool rsh = xsh & 1, wsh = xsh & 2;
  const uint32_t l0 = (uint32_t)gx * (uint32_t)sizeof(T);
  const uint32_t lp = (uint32_t)(rsh ? wrap(gx - 1, geo.L0) : gx) * (uint32_t)sizeof(T);
  const uint32_t lm = (uint32_t)(rsh ? wrap(gx + 1, geo.L0) : gx) * (uint32_t)sizeof(T);
  const uint32_t sp = (uint32_t)(wsh ? gx : wrap(gx + 1, geo.L0)) * (uint32_t)sizeof(T);
  const uint32_t sm = (uint32_t)(wsh ? gx : wrap(gx - 1, geo.L0)) * (uint32_t)sizeof(T);
  // first staged row of population q
  auto f_base = [](int q) constexpr {
    int b = 0;
    for (int k = 1; k < q; k++) b += S::cy[k] > 0 ? 3 : S::cy[k] < 0 ? SH::DOWN : 2;
    return b;
  };
  const uint64_t qbytes = (uint64_t)geo.V * sizeof(T), rbytes = (uint64_t)geo.L0 * sizeof(T);

  // rows of the lattice: `lrow` the next one to load, `srow` the next one to
  // store, stepped instead of reduced modulo L1 in every iteration
  int lrow = ((m0 - HALO) % Lm + Lm) % Lm, srow = m0;
  // masks of rows j to j - 4 and, in flight with fn, of the next; its psi
  uint32_t mn = 0, mk[5] = {};
  double pn = 0;
  auto load_row = [&](T (&f)[Q]) {
    uint64_t base = (uint64_t)pop + (uint64_t)lrow * rbytes;
    if constexpr (WALLS) {
      mn = *(const IDMX_GLOBAL uint32_t*)((const IDMX_GLOBAL char*)sgpr_u64(
                                              (uint64_t)wmask + (uint64_t)lrow * rbytes) + l0);
      pn = *(const IDMX_GLOBAL double*)((const IDMX_GLOBAL char*)sgpr_u64(
                                            (uint64_t)psi_out + (uint64_t)lrow * rbytes) + l0);
    }
    lrow = lrow + 1 == Lm ? 0 : lrow + 1;
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const IDMX_GLOBAL char* b = (const IDMX_GLOBAL char*)sgpr_u64(base);
      f[q] = *(const IDMX_GLOBAL T*)(b + (S::cx[q] > 0 ? lp : S::cx[q] < 0 ? lm : l0));
      base += qbytes;
    }
  };
  auto psi_at = [&](T s) { return psi_of(P.psi_kind, SHIFT ? P.rho0 + s : s); };
  auto sum = [](const T (&f)[Q]) {
    T s = f[0];
#pragma unroll
    for (int q = 1; q < Q; q++) s += f[q];
    return s;
  };

  // The last R + 1 rows of f(0) and f(1) of this thread's column: row r in
  // slot r mod (R + 1), a compile-time index in each of the R + 1 copies of
  // the loop's body, so that no row is moved between registers.
  constexpr int HR = R + 1;
  T fn[Q], fh0[HR][Q], dn0[HR], fh1[HR][Q], dn1[HR], rest0 = T(0), rest1 = T(0);
  load_row(fn);
  // ring slots of row j: psi (mod NS), f*(0) by the rows its populations keep
  int ps = 0, j3 = 0, j2 = 0;
  auto body = [&](auto ph, int j) {
    constexpr int A0 = ph.value;             // slot of f(0) row j
    constexpr int B0 = (A0 + 1) % HR;        // row j - R
    constexpr int A1 = (A0 + HR * 3 - R - 2) % HR;  // f(1) row j - R - 2
    constexpr int B1 = (A1 + 1) % HR;        // row j - 2R - 2
    auto pslot = [&](int d) { return ps + d < 0 ? ps + d + NS : ps + d; };  // row j + d, d <= 0
    auto slot = [&](int q, int d) {  // f*(0) row j + d of population q, -6 <= d <= 0
      if (S::cy[q] < 0 && SH::DOWN == 1) return 0;
      const int n = S::cy[q] > 0 ? 3 : 2;
      const int v = (S::cy[q] > 0 ? j3 : j2) + (d + 3 * n) % n;
      return v >= n ? v - n : v;
    };
    // psi of row j - R - 2 where that is a solid site
    T psolid = T(0);
    if constexpr (WALLS) {
      psolid = ring0[ps][tid + R];
#pragma unroll
      for (int k = 4; k > 0; k--) mk[k] = mk[k - 1];
      mk[0] = mn;
    }
    // psi(0) of row j
    if (j < J - 1) {
      const T pw = pn;
#pragma unroll
      for (int q = 0; q < Q; q++) fh0[A0][q] = fn[q];
      dn0[A0] = sum(fh0[A0]);
      if (j + 1 < J - 1) load_row(fn);
      ring0[ps][tid + R] = WALLS && (mk[0] & (1u << kWallSelf)) ? pw : psi_at(dn0[A0]);
    }
    // f(1) and psi(1) of row j - R - 2
    if (j >= 2 * R + 3) {
#pragma unroll
      for (int q = 0; q < Q; q++)
        fh1[A1][q] = q == 0 ? rest0 : frow[f_base(q) + slot(q, -R - 2)][tid + 1];
      dn1[A1] = sum(fh1[A1]);
      ring1[ps][tid + R] = WALLS && (mk[3] & (1u << kWallSelf)) ? psolid : psi_at(dn1[A1]);
    }
    lds_barrier();
    rest0 = rest1;
    // first step's collision of row j - R
    if (j >= 2 * R && j < J - 1) {
      T gx_, gy_, gz_, fo[Q], u[3];
      iso_grad<ES>([&](int e) { return ring0[pslot(ES::ey[e] - R)][tid + R + ES::ex[e]]; }, gx_,
                   gy_, gz_);
      collide<S, T, SHIFT, COLL, WALLS>(fh0[B0], dn0[B0], gx_, gy_, T(0),
                                        ring0[pslot(-R)][tid + R], PL, fo, u, bx, by);
      rest1 = fo[0];
      // with walls, most waves have no solid site near: one test for the wave
      const uint32_t m = mk[1];
      if (WALLS && __ballot(m != 0) != 0) {
        if (!(m & (1u << kWallSelf))) {
#pragma unroll
          for (int q = 1; q < Q; q++) {
            // aimed at a solid site: back to this one as the opposite
            const int o = opposite<S>(q);
            if (m >> q & 1) frow[f_base(o) + slot(o, -R)][tid + 1] = fo[q];
            else frow[f_base(q) + slot(q, S::cy[q] - R)][tid + 1 + S::cx[q]] = fo[q];
          }
        }
      } else {
#pragma unroll
        for (int q = 1; q < Q; q++)
          frow[f_base(q) + slot(q, S::cy[q] - R)][tid + 1 + S::cx[q]] = fo[q];
      }
    }
    // second step's collision of row j - 2R - 2 (psi(1) of row j - R - 2 + d
    // is in the slot of psi(0) row j + d)
    if (j >= 2 * HALO + 1) {
      T gx_, gy_, gz_, fo[Q], u[3];
      iso_grad<ES>([&](int e) { return ring1[pslot(ES::ey[e] - R)][tid + R + ES::ex[e]]; }, gx_,
                   gy_, gz_);
      const T lpsi = ring1[pslot(-R)][tid + R];
      collide<S, T, SHIFT, COLL, WALLS>(fh1[B1], dn1[B1], gx_, gy_, T(0), lpsi, PL, fo, u, bx,
                                        by);
      if (own && !(WALLS && (mk[4] & (1u << kWallSelf)))) {
        const int sup = srow + 1 == Lm ? 0 : srow + 1, sdn = srow == 0 ? Lm - 1 : srow - 1;
        auto push = [&](int q) {
          st_nt_sbase((uint64_t)pop_swap + q * qbytes +
                          (uint64_t)(S::cy[q] > 0 ? sup : S::cy[q] < 0 ? sdn : srow) * rbytes,
                      S::cx[q] > 0 ? sp : S::cx[q] < 0 ? sm : l0, fo[q]);
        };
        if (WALLS && __ballot(mk[4] != 0) != 0) {
#pragma unroll
          for (int q = 0; q < Q; q++) {
            // back to this site as the opposite: in the x-shifted storage
            // that is kept at x - c_x of the opposite
            if (q > 0 && (mk[4] >> q & 1))
              st_nt_sbase((uint64_t)pop_swap + opposite<S>(q) * qbytes + (uint64_t)srow * rbytes,
                          S::cx[q] == 0 || !wsh
                              ? l0
                              : (uint32_t)wrap(gx + S::cx[q], geo.L0) * (uint32_t)sizeof(T),
                          fo[q]);
            else push(q);
          }
        } else {
#pragma unroll
          for (int q = 0; q < Q; q++) push(q);
        }
        if (WF) {
          const int64_t g = (int64_t)gx + (int64_t)geo.L0 * srow;
          n_out[g] = (double)(SHIFT ? P.rho0 + dn1[B1] : dn1[B1]);
          psi_out[g] = (double)lpsi;
          u_out[g] = (double)u[0];
          u_out[g + geo.V] = (double)u[1];
        }
      }
      srow++;
    }
    lds_barrier();
    ps = ps + 1 == NS ? 0 : ps + 1;
    j3 = j3 == 2 ? 0 : j3 + 1;
    j2 ^= 1;
  };
  for (int j = 0; j < J; j += HR) {
    body(std::integral_constant<int, 0>{}, j);
    if (j + 1 < J) body(std::integral_constant<int, 1>{}, j + 1);
    if constexpr (HR == 3)
      if (j + 2 < J) body(std::integral_constant<int, 2>{}, j + 2);
  }
}

}  // namespace idmx
