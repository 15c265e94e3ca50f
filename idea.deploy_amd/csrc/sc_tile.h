// sc_tile.h -- steps of small lattices: two or four time steps of a D2Q9
// lattice in one launch (k_tile2d), one step of a D3Q19 lattice without a
// march (k_tile3d).
//
// What bounds a small lattice is latency: a step of 128^2 sites moves 2.4 MB
// that stay in L2 and is over in 5.2 us, most of it launch, two memory
// latencies and a barrier. A block here loads a B x B tile with the ring of
// sites that KS steps reach, takes the steps in LDS on a region that shrinks
// by R + 1 sites per side and step (R the reach of the force stencil), and
// pushes the result: one launch and one round trip to memory per KS steps,
// paid for with redundant collisions on the ring (E4, KS = 4: 3.4 times the
// sites of an 8 x 8 tile, 2.0 of a 16 x 16 one; KS = 2: 1.2 of a 24 x 24 one),
// which an otherwise idle chip has room for; from about 10^5 sites the FP64
// vector units bound it. Measured per step against the register step, one
// launch each: E4 128^2 1.73 us (5.10), 256^2 2.3 (6.06), 512^2 6.3 (11.0);
// E8 128^2 2.5 (7.0), 256^2 3.3 (8.2), 620^2 13.7 (26.5), in FP32 7.4 (16.2).
//
// One site per thread: thread t is site (t mod w, t / w) of the stage's
// region of w x w sites, where psi is needed (PW); it collides there unless
// it lies within R of the region's rim.
#pragma once
#include <type_traits>

#include "sc_kernels.h"

namespace idmx {

template <int B, int KS, int R>
struct TileShape {
  // psi of stage s, collisions
  static constexpr int PW(int s) { return B + 2 * ((R + 1) * (KS - 1 - s) + R); }
  static constexpr int CW(int s) { return PW(s) - 2 * R; }
  static constexpr int NT = (PW(0) * PW(0) + 63) / 64 * 64;
  // f* of even and odd stages (that of the last one goes to memory)
  static constexpr int F0 = CW(0) * CW(0), F1 = KS > 2 ? CW(1) * CW(1) : 1;
};

// WALLS: flags 0 and 1 only; the masks and the solid sites' psi (psi_out,
// which keeps them) are read once and kept in LDS, and a site next to a solid
// one takes the population that would stream in from there from its own f*.
// u_out may then be null.
template <class ES, class T, bool SHIFT, int COLL, int B, int KS, bool WF, bool WALLS = false>
__global__ void __launch_bounds__((TileShape<B, KS, ES::R>::NT))
k_tile2d(const T* __restrict__ pop, T* __restrict__ pop_swap, Geom geo, Phys<T> P, int ntx,
         int ntiles, double* __restrict__ n_out, double* psi_out, double* __restrict__ u_out,
         const uint64_t* __restrict__ wmask = nullptr, T bx = T(0), T by = T(0)) {
  using S = D2Q9;
  constexpr int R = ES::R;
  using SH = TileShape<B, KS, R>;
  constexpr int Q = S::Q, NB = NBasis<2>::value;
  constexpr int NTAB = COLL == 2 ? Q : COLL == 1 ? Q * Q + 2 * NB * Q : 1;
  __shared__ T fa[Q][SH::F0], fb[Q][SH::F1];
  __shared__ T pa[SH::PW(0) * SH::PW(0)], pb[SH::PW(1) * SH::PW(1)];
  __shared__ T tab[NTAB];
  // masks and psi of the solid sites of stage 0's region
  constexpr int W0 = WALLS ? SH::PW(0) : 1;
  __shared__ T pwall[W0 * W0];
  __shared__ uint32_t wall[W0 * W0];
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
    // this site in stage 0's region
    const int w0 = WALLS ? (py + (W0 - PW) / 2) * W0 + px + (W0 - PW) / 2 : 0;
    uint32_t m = 0;
    T f[Q], dn = T(0);
    if (in) {
      if constexpr (s == 0) {
        constexpr int D = (R + 1) * (KS - 1) + R;
        const int x = ((x0 - D + px) % geo.L0 + geo.L0) % geo.L0;
        const int y = ((y0 - D + py) % geo.L1 + geo.L1) % geo.L1;
        const int64_t g = (int64_t)y * geo.L0 + x;
#pragma unroll
        for (int q = 0; q < Q; q++) f[q] = pop_ld(pop, q, geo.V, g);
        if constexpr (WALLS) {
          m = (uint32_t)wmask[g];
          wall[w0] = m;
          pwall[w0] = (T)psi_out[g];
        }
      } else {
        if constexpr (WALLS) m = wall[w0];
        // f streamed from the previous stage's f*: its region reaches one
        // site further on every side
#pragma unroll
        for (int q = 0; q < Q; q++)
          f[q] = WALLS && q > 0 && (m >> opposite<S>(q) & 1)
                     ? fin[opposite<S>(q) * fin_n + (py + 1) * IW + px + 1]
                     : fin[q * fin_n + (py + 1 - S::cy[q]) * IW + px + 1 - S::cx[q]];
      }
      dn = f[0];
#pragma unroll
      for (int q = 1; q < Q; q++) dn += f[q];
      psi[tid] = WALLS && (m >> kWallSelf & 1) ? pwall[w0]
                                               : psi_of(P.psi_kind, SHIFT ? P.rho0 + dn : dn);
    }
    __syncthreads();
    if (in && px >= R && px < PW - R && py >= R && py < PW - R) {
      T gx, gy, gz, fo[Q], u[3];
      iso_grad<ES>([&](int e) { return psi[tid + ES::ey[e] * PW + ES::ex[e]]; }, gx, gy, gz);
      const T lpsi = psi[tid];
      collide<S, T, SHIFT, COLL, WALLS>(f, dn, gx, gy, T(0), lpsi, PL, fo, u, bx, by);
      if constexpr (s < KS - 1) {
        const int c = (py - R) * CW + px - R;
#pragma unroll
        for (int q = 0; q < Q; q++) fout[q * fout_n + c] = fo[q];
      } else {
        const int x = x0 + px - R, y = y0 + py - R;
        if (x < geo.L0 && y < geo.L1 && !(WALLS && (m >> kWallSelf & 1))) {
          const int64_t g = (int64_t)x + (int64_t)geo.L0 * y;
          if (WALLS && m != 0) {
            // aimed at a solid site: back to this one as the opposite
#pragma unroll
            for (int q = 0; q < Q; q++) {
              const int xt = wrap(x + S::cx[q], geo.L0), yt = wrap(y + S::cy[q], geo.L1);
              if (q > 0 && (m >> q & 1)) pop_st_nt(pop_swap, opposite<S>(q), geo.V, g, fo[q]);
              else pop_st_nt(pop_swap, q, geo.V, lex(geo, xt, yt, 0), fo[q]);
            }
          } else {
            push_store<S, T>(pop_swap, geo, x, y, 0, fo);
          }
          if (WF) {
            n_out[g] = (double)(SHIFT ? P.rho0 + dn : dn);
            psi_out[g] = (double)lpsi;
            if (!WALLS || u_out) {
              u_out[g] = (double)u[0];
              u_out[g + geo.V] = (double)u[1];
            }
          }
        }
      }
    }
    if constexpr (s < KS - 1) __syncthreads();
  };
  static_assert(KS == 2 || KS == 4, "stages are written out");
  stage(std::integral_constant<int, 0>{}, nullptr, 0, fa[0], SH::F0, pa);
  if constexpr (KS == 4) {
    stage(std::integral_constant<int, 1>{}, fa[0], SH::F0, fb[0], SH::F1, pb);
    stage(std::integral_constant<int, 2>{}, fb[0], SH::F1, fa[0], SH::F0, pa);
  }
  stage(std::integral_constant<int, KS - 1>{}, fa[0], SH::F0, nullptr, 0, pb);
}

// --------------------------------------------------------------------------
// One step of a small D3Q19 lattice, one site per thread: a block loads a
// 16 x 4 x 4 tile and sums the densities of its R-wide halo, all loads
// independent of each other, then collides and pushes. The march of
// k_fused / k_fused_dma reads each population about once, but as a chain of
// H + 2R dependent planes, and a lattice of 10^4 to 10^5 sites leaves no
// second block on a CU to hide them; this step reads 2.5 times the sites
// (R = 1), from L2, in one round trip. Bound by that round trip and the launch
// on 24^3 (7.6 us per step, the march 13.1), by L2 traffic on 48 x 44 x 40
// (E4 FP64 11.6 against 14.1, dense MRT 20.4 against 32.6). 16 x 4 x 4: one
// wave per z plane, four whole 128-byte lines of FP64 per row load.
template <class ES>
struct Tile3Shape {
  static constexpr int R = ES::R, TX = 16, TY = 4, TZ = 4, NT = TX * TY * TZ;
  static constexpr int PX = TX + 2 * R, PY = TY + 2 * R, PZ = TZ + 2 * R;
  static constexpr int SLAB = 2 * R * PX * PY;          // halo sites of the z slabs
  static constexpr int RING = PX * PY - TX * TY;        // of each plane between them
  static constexpr int NH = SLAB + TZ * RING;
  static constexpr int YS = 2 * R * PX;                 // of a ring's y slabs
};

template <class ES, class T, bool SHIFT, int COLL, bool WF>
__global__ void __launch_bounds__(256)
k_tile3d(const T* __restrict__ pop, T* __restrict__ pop_swap, Geom geo, Phys<T> P, int ntx,
         int nty, int ntiles, double* __restrict__ n_out, double* __restrict__ psi_out,
         double* __restrict__ u_out) {
  using S = D3Q19;
  using SH = Tile3Shape<ES>;
  constexpr int Q = S::Q, R = SH::R, PX = SH::PX, PY = SH::PY, NB = NBasis<3>::value;
  constexpr int NTAB = COLL == 2 ? Q : COLL == 1 ? Q * Q + 2 * NB * Q : 1;
  __shared__ T psi[SH::PZ][PY][PX];
  __shared__ T tab[NTAB];
  const int per = gridDim.x >> 3;
  int t = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (t >= ntiles) return;
  const int x0 = t % ntx * SH::TX;
  t /= ntx;
  const int y0 = t % nty * SH::TY, z0 = t / nty * SH::TZ;
  const int tid = threadIdx.x;
  Phys<T> PL = P;
  if constexpr (COLL == 1 || COLL == 2) {
    for (int i = tid; i < NTAB; i += SH::NT) tab[i] = P.mrtA[i];
    PL.mrtA = tab;
    PL.mrtB = COLL == 1 ? tab + Q * Q : nullptr;
    PL.mrtG = COLL == 1 ? tab + Q * Q + NB * Q : nullptr;
  }
  // periodic coordinate, one period out of range at most where the axis is as
  // long as the haloed tile
  auto per1 = [](int v, int L) {
    if (L >= PX) return wrap(v, L);
    return ((v % L) + L) % L;
  };
  const int tx = tid % SH::TX, ty = tid / SH::TX % SH::TY;
  const int tz = __builtin_amdgcn_readfirstlane(tid / (SH::TX * SH::TY));  // one plane per wave
  const int x = x0 + tx, y = y0 + ty, z = z0 + tz;
  const bool own = x < geo.L0 && y < geo.L1 && z < geo.L2;
  const int xw = per1(x, geo.L0), yw = per1(y, geo.L1), zw = per1(z, geo.L2);
  const uint32_t E = (uint32_t)sizeof(T), L0 = (uint32_t)geo.L0, L01 = L0 * (uint32_t)geo.L1;
  const uint64_t qbytes = (uint64_t)geo.V * sizeof(T);
  auto load = [&](uint64_t base, uint32_t off, T (&f)[Q]) {
#pragma unroll
    for (int q = 0; q < Q; q++) {
      f[q] = *(const IDMX_GLOBAL T*)((const IDMX_GLOBAL char*)sgpr_u64(base) + off);
      base += qbytes;
    }
  };
  T f[Q];
  const uint32_t own_off = ((uint32_t)xw + L0 * (uint32_t)yw) * E;
  load((uint64_t)pop + (uint64_t)L01 * (uint32_t)zw * E, own_off, f);
#pragma unroll
  for (int k = 0; k < (SH::NH + SH::NT - 1) / SH::NT; k++) {
    const int h = tid + k * SH::NT;
    if (h < SH::NH) {
      int hx, hy, hz;
      if (h < SH::SLAB) {
        const int p = h / (PX * PY), r = h % (PX * PY);
        hz = p < R ? p : SH::TZ + p;
        hy = r / PX;
        hx = r % PX;
      } else {
        const int k2 = h - SH::SLAB, r = k2 % SH::RING;
        hz = R + k2 / SH::RING;
        if (r < SH::YS) {
          const int p = r / PX;
          hy = p < R ? p : SH::TY + p;
          hx = r % PX;
        } else {
          const int c = (r - SH::YS) % (2 * R);
          hy = R + (r - SH::YS) / (2 * R);
          hx = c < R ? c : SH::TX + c;
        }
      }
      const uint32_t off = ((uint32_t)per1(x0 - R + hx, geo.L0) +
                            L0 * (uint32_t)per1(y0 - R + hy, geo.L1) +
                            L01 * (uint32_t)per1(z0 - R + hz, geo.L2)) * E;
      T fh[Q];
      load((uint64_t)pop, off, fh);
      arrive(fh);
      const T s = pop_sum(fh);
      psi[hz][hy][hx] = psi_of(P.psi_kind, SHIFT ? P.rho0 + s : s);
    }
  }
  const T dn = pop_sum(f);
  const T lpsi = psi_of(P.psi_kind, SHIFT ? P.rho0 + dn : dn);
  psi[tz + R][ty + R][tx + R] = lpsi;
  __syncthreads();
  if (!own) return;
  T gx, gy, gz, fo[Q], u[3];
  iso_grad<ES>(
      [&](int e) { return psi[tz + R + ES::ez[e]][ty + R + ES::ey[e]][tx + R + ES::ex[e]]; }, gx,
      gy, gz);
  collide<S, T, SHIFT, COLL>(f, dn, gx, gy, gz, lpsi, PL, fo, u);
  // push: in-plane offsets per lane, the target plane in the scalar base
  const int xs[3] = {wrap(x - 1, geo.L0), x, wrap(x + 1, geo.L0)};
  const int ys[3] = {wrap(y - 1, geo.L1), y, wrap(y + 1, geo.L1)};
  const int zs[3] = {wrap(z - 1, geo.L2), z, wrap(z + 1, geo.L2)};
#pragma unroll
  for (int q = 0; q < Q; q++)
    st_nt_sbase((uint64_t)pop_swap + q * qbytes + (uint64_t)L01 * (uint32_t)zs[S::cz[q] + 1] * E,
                ((uint32_t)xs[S::cx[q] + 1] + L0 * (uint32_t)ys[S::cy[q] + 1]) * E, fo[q]);
  if (WF) {
    const int64_t g = lex(geo, x, y, z);
    n_out[g] = (double)(SHIFT ? P.rho0 + dn : dn);
    psi_out[g] = (double)lpsi;
    u_out[g] = (double)u[0];
    u_out[g + geo.V] = (double)u[1];
    u_out[g + 2 * geo.V] = (double)u[2];
  }
}

}  // namespace idmx
