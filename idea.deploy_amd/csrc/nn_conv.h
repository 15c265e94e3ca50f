// nn_conv.h -- tiled 3x3 convolution kernels of the warm-start network
// (forward / backward-data, and backward-weight) on BF16 MFMA; NHWC tensors.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace idmx {

typedef short v4i16 __attribute__((ext_vector_type(4)));
typedef float v4f32 __attribute__((ext_vector_type(4)));
typedef uint32_t v2u32 __attribute__((ext_vector_type(2)));
typedef uint32_t v4u32 __attribute__((ext_vector_type(4)));

__device__ inline float bf2f(uint16_t b) {
  return __uint_as_float(((uint32_t)b) << 16);
}
// round to nearest even
__device__ inline uint16_t f2bf(float f) {
  uint32_t u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)(u >> 16);  // inf / nan
  u += 0x7fffu + ((u >> 16) & 1u);
  return (uint16_t)(u >> 16);
}

struct ConvShape {
  int N, H, W, Cin, Cout;
};

// The sums over a weight gradient's parts: dw[i] += sum_b part[b][i] (i < nw),
// db[i - nw] likewise (db may be null), 64 sums per block, its four waves over
// a quarter of the parts each, eight loads in flight.
struct BwdWSum {
  const float* part = nullptr;
  float *dw = nullptr, *db = nullptr;
  int nw = 0, n = 0, parts = 0;
  int nx = 0;  // in a convolution's launch: its own blocks along x
};
__device__ inline void bwd_w_sum(const BwdWSum& t, int block, float* f) {
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6, i = block * 64 + lane;
  float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  if (i < t.n) {
    int b = g;
    for (; b + 28 < t.parts; b += 32)
#pragma unroll
      for (int k = 0; k < 8; k++) v[k] += t.part[(int64_t)(b + 4 * k) * t.n + i];
    for (; b < t.parts; b += 4) v[0] += t.part[(int64_t)b * t.n + i];
  }
  f[threadIdx.x] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  __syncthreads();
  if (g == 0 && i < t.n) {
    const float r = (f[lane] + f[64 + lane]) + (f[128 + lane] + f[192 + lane]);
    if (i < t.nw) t.dw[i] += r;
    else if (t.db) t.db[i - t.nw] += r;
  }
}

// ---------------------------------------------------------------------------
// Forward 3x3 convolution of TP consecutive pixels (in (n, y, x) order) by CT
// tiles of 16 output channels per block; the arithmetic of k_conv3x3_fwd, in
// its order (16 k values per MFMA, k = tap * CIN + ci ascending), so the two
// agree bit for bit. The weights are the MFMA's rows and the pixels its
// columns, so a lane ends with 4 output channels of one pixel (8-byte stores).
//
// Bound by latency at these sizes (a layer of the batch-32 network is 0.3 to
// 1.2 GFLOP and 1 to 25 MB): a wave's weights, at most 144 registers, are
// requested before the rows are staged, so one latency covers both, and the
// loop over taps reads LDS only.
template <int CIN>
struct ConvTile {
  // dwords between pixels in LDS: 16 lanes read 16 consecutive pixels, 8
  // dwords each, and these strides spread them over all 64 banks
  static constexpr int SD = CIN == 8 ? 4 : CIN == 16 ? 8 : CIN == 32 ? 24 : CIN / 2 + 4;
  static constexpr int ZERO = 3 * SD;  // dwords of a zero area
  static constexpr int CTMAX = CIN <= 16 ? 4 : CIN == 32 ? 2 : 1;
  static int rows(int W, int tp) { return (tp + W - 2) / W + 1 + 2; }
  static size_t lds(int W, int tp) {
    return 4 * ((size_t)rows(W, tp) * (W + 2) * SD + ZERO);
  }
};

template <int CIN, int CT, int TP, bool SUM>
__global__ void __launch_bounds__(256)
k_conv3x3_tile(const uint16_t* __restrict__ in, const uint16_t* __restrict__ wt,
               const float* __restrict__ bias, uint16_t* __restrict__ out,
               float* __restrict__ out_f32, ConvShape s, int relu, BwdWSum t) {
  using C = ConvTile<CIN>;
  constexpr int SD = C::SD, K = 9 * CIN, NM = TP / 64;  // 16-pixel tiles per wave
  constexpr int NSL = (K + 15) / 16;                    // MFMAs along k
  extern __shared__ uint32_t lds[];
  // SUM, a backward-data launch: the blocks past its own along x add up the
  // layer's weight gradient (a launch of its own takes 4.4 us: a training step
  // of 32 images 457 us with them, 390 without)
  if (SUM && (int)blockIdx.x >= t.nx) {
    bwd_w_sum(t, (blockIdx.x - t.nx) * gridDim.y + blockIdx.y, (float*)lds);
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int P = s.N * s.H * s.W, W = s.W;
  const int p0 = blockIdx.x * TP;
  const int row0 = p0 / W - 1;  // first staged row, rows counted over all images
  const int nrows = (min(p0 + TP, P) - 1) / W + 1 - row0 + 1;
  const int nr_all = s.N * s.H;
  const int r = lane & 15, kq = lane >> 4;
  const int ct0 = blockIdx.y * CT;

  v4i16 wf[NSL][CT];
#pragma unroll
  for (int c = 0; c < CT; c++) {
    const int co = (ct0 + c) * 16 + r;
    const uint16_t* w = wt + (int64_t)(co < s.Cout ? co : 0) * K + 4 * kq;
#pragma unroll
    for (int i = 0; i < NSL; i++) {
      wf[i][c] = v4i16{0, 0, 0, 0};
      if (co < s.Cout && (K % 16 == 0 || 16 * i + 4 * kq < K)) wf[i][c] = *(const v4i16*)(w + 16 * i);
    }
  }

  // stage the rows, with a zero pixel at both ends, 8 channels per access and
  // U accesses per thread in flight (one at a time: 21 us instead of 16 for
  // 16 -> 16 channels of 128 64 x 64 images)
  constexpr int CH = CIN / 8, U = CIN <= 16 ? 4 : 8;
  const int cols = W + 2, rowlen = cols * CH;
  for (int i = tid; i < C::ZERO; i += 256) lds[i] = 0;
  for (int row = 0, i = tid; row < nrows;) {
    v4u32 v[U];
    int dst[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      while (i >= rowlen) {
        i -= rowlen;
        row++;
      }
      const int x = i / CH - 1, c8 = i % CH, g = row0 + row;
      v[u] = v4u32{0, 0, 0, 0};
      dst[u] = row < nrows ? C::ZERO + (row * cols + x + 1) * SD + c8 * 4 : -1;
      if (row < nrows && g >= 0 && g < nr_all && x >= 0 && x < W)
        v[u] = *(const v4u32*)(in + ((int64_t)g * W + x) * CIN + c8 * 8);
      i += 256;
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (dst[u] >= 0) *(v4u32*)(lds + dst[u]) = v[u];
    while (i >= rowlen && row < nrows) {
      i -= rowlen;
      row++;
    }
  }
  __syncthreads();

  // LDS dword of the pixel left of this lane's pixel in the rows above, at and
  // below it; rows outside its image read the zero area
  uint32_t ra[NM][3];
  int p = p0 + wv * NM * 16 + r;
  int g = p / W, x = p - g * W, y = g % s.H;  // stepped by 16 pixels below
#pragma unroll
  for (int m = 0; m < NM; m++) {
    if (m > 0) {
      p += 16;
      x += 16;
      while (x >= W) {
        x -= W;
        g++;
        y = y + 1 == s.H ? 0 : y + 1;
      }
    }
#pragma unroll
    for (int d = 0; d < 3; d++) {
      const bool ok = p < P && y + d - 1 >= 0 && y + d - 1 < s.H;
      ra[m][d] = ok ? (uint32_t)(C::ZERO + ((g + d - 1 - row0) * cols + x) * SD) : 0u;
      if (CIN >= 16) ra[m][d] += 2 * kq;
    }
  }
  v4f32 acc[NM][CT];
#pragma unroll
  for (int m = 0; m < NM; m++)
#pragma unroll
    for (int c = 0; c < CT; c++) acc[m][c] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < NSL; i++)
#pragma unroll
    for (int m = 0; m < NM; m++) {
      v4i16 a;
      if constexpr (CIN >= 16) {
        const int tap = 16 * i / CIN, c0 = 16 * i % CIN;
        a = *(const v4i16*)(lds + ra[m][tap / 3] + tap % 3 * SD + c0 / 2);
      } else {
        // 8 channels: an MFMA's 16 k values are two taps
        const int tap = 2 * i + (kq >> 1);
        const int dy = tap >= 9 ? 0 : tap / 3, dx = tap >= 9 ? 0 : tap % 3;
        const uint32_t base = dy == 0 ? ra[m][0] : dy == 1 ? ra[m][1] : ra[m][2];
        a = *(const v4i16*)(lds + base + dx * SD + 2 * (kq & 1));
        if (tap >= 9) a = v4i16{0, 0, 0, 0};
      }
#pragma unroll
      for (int c = 0; c < CT; c++)
        acc[m][c] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wf[i][c], a, acc[m][c], 0, 0, 0);
    }
  // D: column = lane % 16 (pixel), rows 4 * (lane / 16) + j (output channels)
#pragma unroll
  for (int m = 0; m < NM; m++) {
    const int64_t p = p0 + (wv * NM + m) * 16 + r;
    if (p >= P) continue;
#pragma unroll
    for (int c = 0; c < CT; c++) {
      const int oc = (ct0 + c) * 16 + 4 * kq;
      v4f32 v = acc[m][c];
      if ((s.Cout & 3) == 0) {
        if (oc >= s.Cout) continue;
        if (bias) v += *(const v4f32*)(bias + oc);
        if (out_f32) *(v4f32*)(out_f32 + p * s.Cout + oc) = v;
        uint16_t h[4];
#pragma unroll
        for (int j = 0; j < 4; j++) h[j] = f2bf(relu ? fmaxf(v[j], 0.f) : v[j]);
        *(v2u32*)(out + p * s.Cout + oc) =
            v2u32{h[0] | (uint32_t)h[1] << 16, h[2] | (uint32_t)h[3] << 16};
      } else {
#pragma unroll
        for (int j = 0; j < 4; j++)
          if (oc + j < s.Cout) {
            float t = v[j] + (bias ? bias[oc + j] : 0.f);
            if (out_f32) out_f32[p * s.Cout + oc + j] = t;
            if (relu) t = fmaxf(t, 0.f);
            out[p * s.Cout + oc + j] = f2bf(t);
          }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Backward-weight: dW[co][tap * CIN + ci] = sum_p dY[p][co] X[p + tap][ci] as
// an MFMA GEMM whose reduction runs over pixels. A block accumulates chunks of
// TPX pixels in registers; its sums go to part[block][co * 9 CIN + k] and are
// added up by bwd_w_sum.
//
// The MFMA wants 4 consecutive pixels of one channel per lane, so both
// operands are staged transposed: X as [ci][row][x] with two zero pixels on
// each side, dY as [co][pixel]. One read of the 8 pixels x - 2 .. x + 5 serves
// the three taps of a row (the taps at x - 1 and x + 1 are 16-bit shifts of
// it).
template <int CIN, int COUT, int TPX>
struct BwdW {
  static constexpr int CI = (CIN + 15) / 16, CO = (COUT + 15) / 16;  // 16 x 16 tiles
  // waves: over input-channel tiles first, then output-channel tiles, then
  // groups of pixels (summed over LDS at the end)
  static constexpr int WI = CI < 4 ? CI : 4;
  static constexpr int WO = 4 / WI < CO ? 4 / WI : CO;
  static constexpr int WP = 4 / (WI * WO);
  static constexpr int NI = CI / WI, NO = CO / WO;  // tiles per wave
  // dwords of a channel's rows: 4 mod 8, so that 16 channels fall on 16
  // different quads of banks
  static int plane(int W, int rows) { return ((rows * ((W + 4) / 2)) + 7) / 8 * 8 + 4; }
  static constexpr int YP = TPX / 2 + 4;  // dwords of a channel of dY
  static int rows(int W) { return (TPX + W - 1) / W + 2; }
  static size_t lds(int W) {
    const size_t st = 4 * (4 + (size_t)CIN * plane(W, rows(W)) + (size_t)COUT * YP);
    const size_t red = WP > 1 ? (size_t)3 * 64 * 4 * 9 * NI * NO * 4 : 0;
    return st > red ? st : red;
  }
};

// 8 bf16 values of g where those of y are positive, else 0
__device__ __forceinline__ v4u32 relu_mask(v4u32 y, v4u32 g) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const uint32_t lo = __uint_as_float(y[i] << 16) > 0.f ? 0xffffu : 0u;
    const uint32_t hi = __uint_as_float(y[i] & 0xffff0000u) > 0.f ? 0xffff0000u : 0u;
    g[i] &= lo | hi;
  }
  return g;
}

// 16-bit pairs (hi of a, lo of b) -> dword
__device__ __forceinline__ uint32_t mid16(uint32_t a, uint32_t b) { return (a >> 16) | (b << 16); }

// With y (the layer's ReLU output) dY is masked by y > 0 first, in place: a
// block stages every channel of its pixels, each exactly once. The blocks past
// the first `blocks` write the weights for the backward-data pass instead, the
// transposed, tap-flipped kernel wd[ci][tap' Cout + co] =
// w[co][(8 - tap') Cin + ci] in bf16.
template <int CIN, int COUT, int TPX>
__global__ void __launch_bounds__(256)
k_conv3x3_bwd_w_tile(const uint16_t* __restrict__ in, uint16_t* __restrict__ dy,
                     const uint16_t* __restrict__ y, float* __restrict__ part, ConvShape s,
                     int nchunks, int blocks, const float* __restrict__ w,
                     uint16_t* __restrict__ wd) {
  using B = BwdW<CIN, COUT, TPX>;
  constexpr int NI = B::NI, NO = B::NO, YP = B::YP;
  extern __shared__ uint32_t lds[];
  if ((int)blockIdx.x >= blocks) {
    const int i = (blockIdx.x - blocks) * 256 + threadIdx.x;
    if (i < COUT * 9 * CIN) {
      const int ci = i / (9 * COUT), rem = i % (9 * COUT), tp = rem / COUT, co = rem % COUT;
      wd[i] = f2bf(w[(int64_t)co * 9 * CIN + (8 - tp) * CIN + ci]);
    }
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int W = s.W, H = s.H, P = s.N * H * W;
  const int rw = (W + 4) / 2, nrows = TPX / W + 2, plane = ((nrows * rw) + 7) / 8 * 8 + 4;
  uint32_t* xs = lds + 4;
  uint32_t* ys = xs + CIN * plane;
  const int r = lane & 15, kq = lane >> 4;
  const int wi = wv % B::WI, wo = wv / B::WI % B::WO, wp = wv / (B::WI * B::WO);
  const int nr_all = s.N * H;
  const int lq4 = 31 - __builtin_clz(W / 4);
  if (tid < 4) lds[tid] = 0;
  // the zero pixels at both ends of every staged row
  for (int i = tid; i < CIN * nrows; i += 256) {
    const int c = i / nrows, row = i - c * nrows;
    xs[c * plane + row * rw] = 0;
    xs[c * plane + row * rw + rw - 1] = 0;
  }
  v4f32 acc[NI][3][3][NO];
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
      for (int o = 0; o < NO; o++) acc[i][t / 3][t % 3][o] = {0.f, 0.f, 0.f, 0.f};
  float bsum = 0.f;

  for (int ch = blockIdx.x; ch < nchunks; ch += blocks) {
    const int p0 = ch * TPX, row0 = p0 / W - 1;
    __syncthreads();
    // X: 4 pixels x 8 channels per thread and round, transposed in registers
    // (row and column by shifts: W / 4 is a power of two, as W divides TPX)
    constexpr int CH = CIN / 8;
    for (int i = tid; i < (nrows << lq4) * CH; i += 256) {
      const int c8 = i % CH, t = i / CH;
      const int x4 = t & ((1 << lq4) - 1), row = t >> lq4, g = row0 + row;
      v4u32 v[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        v[k] = v4u32{0, 0, 0, 0};
        if (g >= 0 && g < nr_all)
          v[k] = *(const v4u32*)(in + ((int64_t)g * W + 4 * x4 + k) * CIN + c8 * 8);
      }
#pragma unroll
      for (int c = 0; c < 8; c++) {
        const uint32_t sh = (c & 1) * 16;
        const uint32_t a = (v[0][c / 2] >> sh & 0xffffu) | (v[1][c / 2] >> sh << 16);
        const uint32_t b = (v[2][c / 2] >> sh & 0xffffu) | (v[3][c / 2] >> sh << 16);
        uint32_t* d = xs + (c8 * 8 + c) * plane + row * rw + 1 + 2 * x4;
        d[0] = a;
        d[1] = b;
      }
    }
    if constexpr (COUT % 8 == 0) {
      constexpr int CO8 = COUT / 8;
      for (int i = tid; i < TPX / 4 * CO8; i += 256) {
        const int c8 = i % CO8, p4 = i / CO8;
        v4u32 v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) {
          v[k] = v4u32{0, 0, 0, 0};
          if (p0 + 4 * p4 + k < P) {
            const int64_t o = (int64_t)(p0 + 4 * p4 + k) * COUT + c8 * 8;
            v[k] = *(const v4u32*)(dy + o);
            if (y) {
              v[k] = relu_mask(*(const v4u32*)(y + o), v[k]);
              *(v4u32*)(dy + o) = v[k];
            }
          }
        }
#pragma unroll
        for (int c = 0; c < 8; c++) {
          const uint32_t sh = (c & 1) * 16;
          uint32_t* d = ys + (c8 * 8 + c) * YP + 2 * p4;
          d[0] = (v[0][c / 2] >> sh & 0xffffu) | (v[1][c / 2] >> sh << 16);
          d[1] = (v[2][c / 2] >> sh & 0xffffu) | (v[3][c / 2] >> sh << 16);
        }
      }
    } else {
      for (int i = tid; i < TPX * COUT; i += 256) {
        const int c = i % COUT, p = i / COUT;
        const int64_t o = (int64_t)(p0 + p) * COUT + c;
        uint16_t v = p0 + p < P ? dy[o] : (uint16_t)0;
        if (y && p0 + p < P) {
          v = bf2f(y[o]) > 0.f ? v : (uint16_t)0;
          dy[o] = v;
        }
        ((uint16_t*)(ys + c * YP))[p] = v;
      }
    }
    __syncthreads();
    // bias gradient: the wave's share of the chunk's dY, channel tid % COUT
    {
      constexpr int TPC = 256 / COUT;  // threads per channel
      const int c = tid % COUT, k = tid / COUT;
      if (k < TPC)
        for (int i = k; i < TPX / 2; i += TPC) {
          const uint32_t v = ys[c * YP + i];
          bsum += bf2f((uint16_t)v) + bf2f((uint16_t)(v >> 16));
        }
    }
    for (int px = wp * 16; px < TPX; px += 16 * B::WP) {
      const int pq = px + 4 * kq, p = p0 + pq;  // this lane's 4 pixels
      const int g = p / W, x = p - g * W, yr = g % H;
      v4i16 a[NO];
#pragma unroll
      for (int o = 0; o < NO; o++) {
        const int co = (wo * NO + o) * 16 + r;
        a[o] = *(const v4i16*)(ys + (COUT % 16 == 0 || co < COUT ? co : COUT - 1) * YP + pq / 2);
      }
#pragma unroll
      for (int i = 0; i < NI; i++) {
        const int ci = (wi * NI + i) * 16 + r;
        const uint32_t cb = 4 + (CIN % 16 == 0 || ci < CIN ? ci : ci - CIN) * plane + x / 2;
#pragma unroll
        for (int d = 0; d < 3; d++) {
          const bool ok = p < P && yr + d - 1 >= 0 && yr + d - 1 < H;
          const uint32_t* src = lds + (ok ? cb + (g + d - 1 - row0) * rw : 0u);
          const uint32_t w0 = src[0], w1 = src[1], w2 = src[2], w3 = src[3];
          const uint32_t m01 = mid16(w0, w1), m12 = mid16(w1, w2), m23 = mid16(w2, w3);
          v4i16 b[3];
          b[0] = __builtin_bit_cast(v4i16, (v2u32{m01, m12}));
          b[1] = __builtin_bit_cast(v4i16, (v2u32{w1, w2}));
          b[2] = __builtin_bit_cast(v4i16, (v2u32{m12, m23}));
#pragma unroll
          for (int t = 0; t < 3; t++)
#pragma unroll
            for (int o = 0; o < NO; o++)
              acc[i][d][t][o] =
                  __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a[o], b[t], acc[i][d][t][o], 0, 0, 0);
        }
      }
    }
  }
  __syncthreads();
  constexpr int KK = 9 * CIN;
  float* out = part + (int64_t)blockIdx.x * (COUT * KK + COUT);
  // bias partial: over the threads of a channel, through LDS
  {
    float* f = (float*)lds;
    f[tid] = bsum;
    __syncthreads();
    if (tid < COUT) {
      float t = 0.f;
      for (int k = 0; k < 256 / COUT; k++) t += f[tid + k * COUT];
      out[COUT * KK + tid] = t;
    }
    __syncthreads();
  }
  if constexpr (B::WP > 1) {
    // groups of pixels: all but the first hand their sums over
    v4f32* f = (v4f32*)lds;
    constexpr int T = 9 * NI * NO;
    if (wp > 0)
#pragma unroll
      for (int t = 0; t < T; t++)
        f[((wv - B::WI * B::WO) * T + t) * 64 + lane] =
            acc[t / (9 * NO)][t / (3 * NO) % 3][t / NO % 3][t % NO];
    __syncthreads();
    if (wp > 0) return;
#pragma unroll
    for (int t = 0; t < T; t++)
#pragma unroll
      for (int k = 1; k < B::WP; k++)
        acc[t / (9 * NO)][t / (3 * NO) % 3][t / NO % 3][t % NO] +=
            f[((wv + (k - 1) * B::WI * B::WO) * T + t) * 64 + lane];
  }
#pragma unroll
  for (int i = 0; i < NI; i++)
#pragma unroll
    for (int t = 0; t < 9; t++)
#pragma unroll
      for (int o = 0; o < NO; o++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const int co = (wo * NO + o) * 16 + 4 * kq + j, ci = (wi * NI + i) * 16 + r;
          if (co < COUT && ci < CIN) out[co * KK + t * CIN + ci] = acc[i][t / 3][t % 3][o][j];
        }
}

__global__ void __launch_bounds__(256) k_conv_bwd_w_sum(BwdWSum t) {
  __shared__ float f[256];
  bwd_w_sum(t, blockIdx.x, f);
}

}  // namespace idmx
