// nn.hip -- kernels of the warm-start network (a small U-Net) for gfx950:
// 3x3 convolutions as implicit GEMMs on BF16 MFMA (v_mfma_f32_16x16x16_bf16)
// with FP32 accumulation, forward, backward-data and backward-weight, and
// the elementwise pieces (ReLU backward, 2x2 average pool, nearest 2x
// upsample, channel concat/split, MSE loss, Adam, casts, bilinear resize to
// the lattice). No reference counterpart: idpy has no learned component.
//
// Tensors are NHWC. Activations and weights used by the MFMA are bf16
// (stored as uint16 bit patterns); master weights, gradients and the loss
// are FP32. Conv weights are [Cout][9*Cin] with k = tap*Cin + ci,
// tap = 3*ky + kx. Layers of 8, 16, 32, 64 or 128 channels run the tiled
// kernels of nn_conv.h, the convolutions here take the other shapes: when
// Cin is a multiple of 4 a lane's MFMA K slice is 4
// channels of one tap (vector loads); other channel counts are handled
// element by element.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "internal.h"
#include "nn_conv.h"

namespace idmx {

// ---------------------------------------------------------------------------
// Forward 3x3 convolution, stride 1, zero padding 1:
//   out[p][co] = act(bias[co] + sum_k A[p][k] * Wt[co][k]),
//   A[p][k] = in[n, y+ky-1, x+kx-1, ci] (im2col, never materialised).
// One wave computes a 16 (pixels) x 16 (output channels) tile; K advances
// 16 per MFMA (4 per lane: 4 consecutive input channels of one tap).
// MFMA 16x16x16 lane layout: A row = lane%16, k = 4*(lane/16)+j; B column =
// lane%16, same k; D column = lane%16, rows 4*(lane/16)+j.
// out_f32 (optional) receives the pre-activation FP32 values.
__global__ void __launch_bounds__(256)
k_conv3x3_fwd(const uint16_t* __restrict__ in, const uint16_t* __restrict__ wt,
              const float* __restrict__ bias, uint16_t* __restrict__ out,
              float* __restrict__ out_f32, ConvShape s, int relu) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int P = s.N * s.H * s.W;
  const int ptiles = (P + 15) / 16;
  const int ctiles = (s.Cout + 15) / 16;
  if (wave >= ptiles * ctiles) return;
  const int pt = wave % ptiles, ct = wave / ptiles;
  const int r = lane & 15, kq = lane >> 4;
  const int p = pt * 16 + r;  // A row (pixel)
  const bool pvalid = p < P;
  const int n = pvalid ? p / (s.H * s.W) : 0;
  const int yx = pvalid ? p % (s.H * s.W) : 0;
  const int y = yx / s.W, x = yx % s.W;
  const int co = ct * 16 + r;  // B column
  const bool cvalid = co < s.Cout;
  const int K = 9 * s.Cin;
  const bool vec4 = (s.Cin & 3) == 0;
  v4f32 acc = {0.f, 0.f, 0.f, 0.f};
  for (int k0 = 0; k0 < K; k0 += 16) {
    const int k = k0 + 4 * kq;
    v4i16 a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
    if (vec4) {
      // Cin % 4 == 0: the 4 k values of a lane are 4 channels of one tap
      if (k < K) {
        const int tap = k / s.Cin, ci = k % s.Cin;
        const int yy = y + tap / 3 - 1, xx = x + tap % 3 - 1;
        if (pvalid && yy >= 0 && yy < s.H && xx >= 0 && xx < s.W) {
          const uint16_t* src = in + (((int64_t)n * s.H + yy) * s.W + xx) * s.Cin + ci;
#pragma unroll
          for (int j = 0; j < 4; j++) a[j] = (short)src[j];
        }
        if (cvalid) {
          const uint16_t* wsrc = wt + (int64_t)co * K + k;
#pragma unroll
          for (int j = 0; j < 4; j++) b[j] = (short)wsrc[j];
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int kk = k + j;
        if (kk < K) {
          const int tap = kk / s.Cin, ci = kk % s.Cin;
          const int yy = y + tap / 3 - 1, xx = x + tap % 3 - 1;
          if (pvalid && yy >= 0 && yy < s.H && xx >= 0 && xx < s.W)
            a[j] = (short)in[(((int64_t)n * s.H + yy) * s.W + xx) * s.Cin + ci];
          if (cvalid) b[j] = (short)wt[(int64_t)co * K + kk];
        }
      }
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  }
  // D: column = lane%16 (output channel), rows 4*(lane/16)+j (pixels)
  const int oc = ct * 16 + (lane & 15);
  if (oc < s.Cout) {
    const float bv = bias ? bias[oc] : 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int op = pt * 16 + 4 * kq + j;
      if (op < P) {
        float v = acc[j] + bv;
        if (out_f32) out_f32[(int64_t)op * s.Cout + oc] = v;
        if (relu) v = fmaxf(v, 0.f);
        out[(int64_t)op * s.Cout + oc] = f2bf(v);
      }
    }
  }
}

// Backward-weight: dW[co][k] += sum_p dY[p][co] * A[p][k] over a chunk of
// pixels per wave (split over pixels, FP32 atomics into dW). MFMA rows are
// output channels, columns are k, the reduction runs over 16 pixels per
// instruction (4 per lane).
__global__ void __launch_bounds__(256)
k_conv3x3_bwd_w(const uint16_t* __restrict__ in, const uint16_t* __restrict__ dy,
                float* __restrict__ dw, ConvShape s, int pchunk) {
  const int lane = threadIdx.x & 63;
  const int wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  const int P = s.N * s.H * s.W;
  const int K = 9 * s.Cin;
  const int ctiles = (s.Cout + 15) / 16, ktiles = (K + 15) / 16;
  const int nchunks = (P + pchunk - 1) / pchunk;
  if (wave >= ctiles * ktiles * nchunks) return;
  int t = wave;
  const int kt = t % ktiles;
  t /= ktiles;
  const int ct = t % ctiles;
  const int ch = t / ctiles;
  const int r = lane & 15, kq = lane >> 4;
  const int co = ct * 16 + r;  // A row
  const int k = kt * 16 + r;   // B column
  const bool cvalid = co < s.Cout, kvalid = k < K;
  const int tap = kvalid ? k / s.Cin : 0, ci = kvalid ? k % s.Cin : 0;
  const int dy_ = tap / 3 - 1, dx_ = tap % 3 - 1;
  v4f32 acc = {0.f, 0.f, 0.f, 0.f};
  const int pbeg = ch * pchunk, pend = min(P, pbeg + pchunk);
  for (int p0 = pbeg; p0 < pend; p0 += 16) {
    v4i16 a = {0, 0, 0, 0}, b = {0, 0, 0, 0};
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int p = p0 + 4 * kq + j;
      if (p < pend) {
        if (cvalid) a[j] = (short)dy[(int64_t)p * s.Cout + co];
        if (kvalid) {
          const int n = p / (s.H * s.W), yx = p % (s.H * s.W);
          const int yy = yx / s.W + dy_, xx = yx % s.W + dx_;
          if (yy >= 0 && yy < s.H && xx >= 0 && xx < s.W)
            b[j] = (short)in[(((int64_t)n * s.H + yy) * s.W + xx) * s.Cin + ci];
        }
      }
    }
    acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  }
  const int kc = kt * 16 + (lane & 15);
  if (kc < K) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int oc = ct * 16 + 4 * kq + j;
      if (oc < s.Cout) atomicAdd(dw + (int64_t)oc * K + kc, acc[j]);
    }
  }
}

// Weights for the backward-data pass: the transposed, tap-flipped kernel
// Wd[ci][tap'*Cout + co] = Wt[co][(8 - tap')*Cin + ci], in bf16.
__global__ void k_conv_flip_weights(const float* __restrict__ w, uint16_t* __restrict__ wd,
                                    int Cin, int Cout) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  const int total = Cin * 9 * Cout;
  if (i >= total) return;
  const int ci = i / (9 * Cout), rem = i % (9 * Cout);
  const int tp = rem / Cout, co = rem % Cout;
  wd[i] = f2bf(w[(int64_t)co * 9 * Cin + (8 - tp) * Cin + ci]);
}

// dX = dY * (Y > 0) on bf16 tensors (ReLU backward from the stored output).
__global__ void k_relu_bwd(const uint16_t* __restrict__ y, const uint16_t* __restrict__ dy,
                           uint16_t* __restrict__ dx, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    dx[i] = bf2f(y[i]) > 0.f ? dy[i] : (uint16_t)0;
}

// db[c] = sum_p dY[p][c] (FP32)
__global__ void k_bias_grad(const uint16_t* __restrict__ dy, float* __restrict__ db, int P,
                            int C) {
  const int c = blockIdx.x;
  float s = 0.f;
  for (int p = threadIdx.x; p < P; p += blockDim.x) s += bf2f(dy[(int64_t)p * C + c]);
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  __shared__ float part[16];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.f;
    for (int k = 0; k < (int)(blockDim.x >> 6); k++) t += part[k];
    db[c] += t;
  }
}

// 2x2 average pool (H, W even) and its backward.
__global__ void k_pool2_fwd(const uint16_t* __restrict__ x, uint16_t* __restrict__ y, int N,
                            int H, int W, int C) {
  const int64_t total = (int64_t)N * (H / 2) * (W / 2) * C;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int c = i % C;
    int64_t t = i / C;
    const int xo = t % (W / 2);
    t /= (W / 2);
    const int yo = t % (H / 2);
    const int n = t / (H / 2);
    float s = 0.f;
    for (int dy = 0; dy < 2; dy++)
      for (int dx = 0; dx < 2; dx++)
        s += bf2f(x[(((int64_t)n * H + 2 * yo + dy) * W + 2 * xo + dx) * C + c]);
    y[i] = f2bf(0.25f * s);
  }
}

__global__ void k_pool2_bwd(const uint16_t* __restrict__ dy, uint16_t* __restrict__ dx, int N,
                            int H, int W, int C) {
  const int64_t total = (int64_t)N * H * W * C;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int c = i % C;
    int64_t t = i / C;
    const int x = t % W;
    t /= W;
    const int y = t % H;
    const int n = t / H;
    dx[i] = f2bf(0.25f * bf2f(dy[(((int64_t)n * (H / 2) + y / 2) * (W / 2) + x / 2) * C + c]));
  }
}

// Nearest 2x upsample of x (N, H, W, C) into channels [c0, c0 + C) of y
// (N, 2H, 2W, Cy), and its backward (sum of the 4 children).
__global__ void k_up2_fwd(const uint16_t* __restrict__ x, uint16_t* __restrict__ y, int N,
                          int H, int W, int C, int Cy, int c0) {
  const int64_t total = (int64_t)N * 2 * H * 2 * W * C;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int c = i % C;
    int64_t t = i / C;
    const int xo = t % (2 * W);
    t /= (2 * W);
    const int yo = t % (2 * H);
    const int n = t / (2 * H);
    y[(((int64_t)n * 2 * H + yo) * 2 * W + xo) * Cy + c0 + c] =
        x[(((int64_t)n * H + yo / 2) * W + xo / 2) * C + c];
  }
}

__global__ void k_up2_bwd(const uint16_t* __restrict__ dy, uint16_t* __restrict__ dx, int N,
                          int H, int W, int C, int Cy, int c0) {
  const int64_t total = (int64_t)N * H * W * C;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int c = i % C;
    int64_t t = i / C;
    const int x = t % W;
    t /= W;
    const int y = t % H;
    const int n = t / H;
    float s = 0.f;
    for (int a = 0; a < 2; a++)
      for (int b = 0; b < 2; b++)
        s += bf2f(dy[(((int64_t)n * 2 * H + 2 * y + a) * 2 * W + 2 * x + b) * Cy + c0 + c]);
    dx[i] = f2bf(s);
  }
}

// Copy channels: y[..., cy0 + c] = x[..., cx0 + c] for c < C (concat / split).
__global__ void k_copy_channels(const uint16_t* __restrict__ x, uint16_t* __restrict__ y,
                                int64_t P, int Cx, int cx0, int Cy, int cy0, int C) {
  const int64_t total = P * C;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * blockDim.x) {
    const int c = i % C;
    const int64_t p = i / C;
    y[p * Cy + cy0 + c] = x[p * Cx + cx0 + c];
  }
}

// Elementwise add of bf16 tensors into FP32 accumulation and back:
// y = bf16(a + b).
__global__ void k_add_bf16(const uint16_t* __restrict__ a, const uint16_t* __restrict__ b,
                           uint16_t* __restrict__ y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = f2bf(bf2f(a[i]) + bf2f(b[i]));
}

// ---------------------------------------------------------------------------
// The same on 8 channels (16 bytes) per thread, for channel counts that are
// multiples of 8 on 16-byte aligned tensors; sums in the same order. The
// scalar kernels above spend their time on index divisions (upsample into the
// concatenated tensor of the 128-image batch: 38.9 us, 6 TB/s would be 11).
struct F8 {
  float v[8];
};
__device__ inline F8 ld8(const uint16_t* p) {
  const v4u32 u = *(const v4u32*)p;
  F8 f;
#pragma unroll
  for (int k = 0; k < 4; k++) {
    f.v[2 * k] = __uint_as_float(u[k] << 16);
    f.v[2 * k + 1] = __uint_as_float(u[k] & 0xffff0000u);
  }
  return f;
}
__device__ inline void st8(uint16_t* p, const F8& f) {
  v4u32 u;
#pragma unroll
  for (int k = 0; k < 4; k++) u[k] = f2bf(f.v[2 * k]) | (uint32_t)f2bf(f.v[2 * k + 1]) << 16;
  *(v4u32*)p = u;
}

__global__ void __launch_bounds__(256)
k_relu_bwd8(const uint16_t* __restrict__ y, const uint16_t* dy, uint16_t* dx, int64_t n8) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n8; i += (int64_t)gridDim.x * 256)
    *(v4u32*)(dx + 8 * i) = relu_mask(*(const v4u32*)(y + 8 * i), *(const v4u32*)(dy + 8 * i));
}

__global__ void __launch_bounds__(256)
k_pool2_fwd8(const uint16_t* __restrict__ x, uint16_t* __restrict__ y, int rows, int Wo, int C8) {
  // rows: N * H / 2 output rows of Wo pixels; a block takes whole rows
  const int C = C8 * 8;
  for (int row = blockIdx.x; row < rows; row += gridDim.x)
    for (int i = threadIdx.x; i < Wo * C8; i += 256) {
      const int xo = i / C8, c = (i - xo * C8) * 8;
      const uint16_t* p = x + ((int64_t)(2 * row) * 2 * Wo + 2 * xo) * C + c;
      const F8 a = ld8(p), b = ld8(p + C), d = ld8(p + (int64_t)2 * Wo * C),
               e = ld8(p + (int64_t)2 * Wo * C + C);
      F8 o;
#pragma unroll
      for (int k = 0; k < 8; k++) o.v[k] = 0.25f * (((a.v[k] + b.v[k]) + d.v[k]) + e.v[k]);
      st8(y + ((int64_t)row * Wo + xo) * C + c, o);
    }
}

// dx = bf16(bf16(dpool / 4) + dcat[..., c0 + c]): gradient of a tensor that
// feeds the pool and channels [c0, c0 + C) of a concatenated one.
__global__ void __launch_bounds__(256)
k_pool2_bwd_add8(const uint16_t* __restrict__ dpool, const uint16_t* __restrict__ dcat,
                 uint16_t* __restrict__ dx, int rows, int W, int C8, int Cc, int c0) {
  const int C = C8 * 8;
  for (int row = blockIdx.x; row < rows; row += gridDim.x)
    for (int i = threadIdx.x; i < W * C8; i += 256) {
      const int x = i / C8, c = (i - x * C8) * 8;
      const F8 a = ld8(dpool + ((int64_t)(row / 2) * (W / 2) + x / 2) * C + c);
      const F8 b = ld8(dcat + ((int64_t)row * W + x) * Cc + c0 + c);
      F8 o;
#pragma unroll
      for (int k = 0; k < 8; k++) o.v[k] = bf2f(f2bf(0.25f * a.v[k])) + b.v[k];
      st8(dx + ((int64_t)row * W + x) * C + c, o);
    }
}

// y = [nearest 2x upsample of x, skip]: rows N * 2H of 2W pixels.
__global__ void __launch_bounds__(256)
k_cat_up2_8(const uint16_t* __restrict__ x, const uint16_t* __restrict__ skip,
            uint16_t* __restrict__ y, int rows, int W, int C8, int S8) {
  const int T8 = C8 + S8;
  for (int row = blockIdx.x; row < rows; row += gridDim.x)
    for (int i = threadIdx.x; i < 2 * W * T8; i += 256) {
      const int xo = i / T8, c = i - xo * T8;
      const uint16_t* src = c < C8 ? x + (((int64_t)(row / 2) * W + xo / 2) * C8 + c) * 8
                                   : skip + (((int64_t)row * 2 * W + xo) * S8 + c - C8) * 8;
      *(v4u32*)(y + (((int64_t)row * 2 * W + xo) * T8 + c) * 8) = *(const v4u32*)src;
    }
}

__global__ void __launch_bounds__(256)
k_up2_bwd8(const uint16_t* __restrict__ dy, uint16_t* __restrict__ dx, int rows, int W, int C8,
           int Cy, int c0) {
  const int C = C8 * 8;
  for (int row = blockIdx.x; row < rows; row += gridDim.x)
    for (int i = threadIdx.x; i < W * C8; i += 256) {
      const int x = i / C8, c = (i - x * C8) * 8;
      const uint16_t* p = dy + ((int64_t)(2 * row) * 2 * W + 2 * x) * Cy + c0 + c;
      const F8 a = ld8(p), b = ld8(p + Cy), d = ld8(p + (int64_t)2 * W * Cy),
               e = ld8(p + (int64_t)2 * W * Cy + Cy);
      F8 o;
#pragma unroll
      for (int k = 0; k < 8; k++) o.v[k] = ((a.v[k] + b.v[k]) + d.v[k]) + e.v[k];
      st8(dx + ((int64_t)row * W + x) * C + c, o);
    }
}

// MSE loss of FP32 prediction vs FP32 target; grad = 2 (pred - target) / n
// in bf16; per-block partial losses in part.
__global__ void __launch_bounds__(256)
k_mse(const float* __restrict__ pred, const float* __restrict__ tgt, uint16_t* __restrict__ grad,
      float* __restrict__ part, int64_t n) {
  float s = 0.f;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x) {
    const float d = pred[i] - tgt[i];
    s += d * d;
    grad[i] = f2bf(2.f * d / (float)n);
  }
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o);
  __shared__ float ps[4];
  if ((threadIdx.x & 63) == 0) ps[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x == 0) part[blockIdx.x] = (ps[0] + ps[1] + ps[2] + ps[3]) / (float)n;
}

// Adam on FP32 master weights; refreshes the bf16 copy; zeroes the gradient.
__device__ __forceinline__ void adam_one(float* __restrict__ w, float* __restrict__ g,
                                         float* __restrict__ m, float* __restrict__ v,
                                         uint16_t* __restrict__ wb, int64_t i, float lr, float b1,
                                         float b2, float eps, float c1, float c2) {
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.f - b1) * gi;
  const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  const float wi = w[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  w[i] = wi;
  if (wb) wb[i] = f2bf(wi);
  g[i] = 0.f;
}

__global__ void k_adam(float* __restrict__ w, float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, uint16_t* __restrict__ wb, int64_t n, float lr,
                       float b1, float b2, float eps, float c1, float c2) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    adam_one(w, g, m, v, wb, i, lr, b1, b2, eps, c1, c2);
}

// The same for up to 32 tensors in one launch: block b works on the tensor
// whose first block is the last one not after b.
struct AdamSet {
  static constexpr int MAX = 32;
  float *w[MAX], *g[MAX], *m[MAX], *v[MAX];
  uint16_t* wb[MAX];
  int64_t n[MAX];
  int first[MAX + 1];
  int count;
};
__global__ void __launch_bounds__(256)
k_adam_set(AdamSet t, float lr, float b1, float b2, float eps, float c1, float c2) {
  int k = 0;
  while (k + 1 < t.count && (int)blockIdx.x >= t.first[k + 1]) k++;
  const int nb = t.first[k + 1] - t.first[k];
  for (int64_t i = (int64_t)(blockIdx.x - t.first[k]) * 256 + threadIdx.x; i < t.n[k];
       i += (int64_t)nb * 256)
    adam_one(t.w[k], t.g[k], t.m[k], t.v[k], t.wb[k], i, lr, b1, b2, eps, c1, c2);
}

__global__ void k_f32_to_bf16(const float* __restrict__ x, uint16_t* __restrict__ y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = f2bf(x[i]);
}

__global__ void k_bf16_to_f32(const uint16_t* __restrict__ x, float* __restrict__ y, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (int64_t)gridDim.x * blockDim.x)
    y[i] = bf2f(x[i]);
}

// Bilinear resize of one S x S FP32 image (pixel centres at (i + 0.5) S/L
// ... in lattice units) to an L x L FP64 lattice field, with a constant
// added (mass correction).
__global__ void k_resize_to_lattice(const float* __restrict__ img, int S, double* __restrict__ n,
                                    int L, double add) {
  const int64_t V = (int64_t)L * L;
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g < V;
       g += (int64_t)gridDim.x * blockDim.x) {
    const int x = g % L, y = g / L;
    const float fx = ((x + 0.5f) * S) / L - 0.5f, fy = ((y + 0.5f) * S) / L - 0.5f;
    int x0 = (int)floorf(fx), y0 = (int)floorf(fy);
    const float ax = fx - x0, ay = fy - y0;
    const int x1 = min(max(x0 + 1, 0), S - 1), y1 = min(max(y0 + 1, 0), S - 1);
    x0 = min(max(x0, 0), S - 1);
    y0 = min(max(y0, 0), S - 1);
    const float v = (1 - ay) * ((1 - ax) * img[y0 * S + x0] + ax * img[y0 * S + x1]) +
                    ay * ((1 - ax) * img[y1 * S + x0] + ax * img[y1 * S + x1]);
    n[g] = (double)v + add;
  }
}

inline unsigned g1(int64_t n, int bs = 256) {
  return (unsigned)std::max<int64_t>(1, std::min<int64_t>((n + bs - 1) / bs, 65536));
}

inline bool aligned(const void* p, size_t n) { return ((uintptr_t)p & (n - 1)) == 0; }

template <int CIN, int TP>
hipError_t conv_tile_ct(idmx_ctx_s* c, const void* in, const void* wt, const float* bias,
                        void* out, float* out_f32, const ConvShape& s, int relu, int ct,
                        BwdWSum t) {
  const int P = s.N * s.H * s.W, cots = (s.Cout + 15) / 16;
  t.nx = (P + TP - 1) / TP;
  const int gy = cots / ct, sums = t.part ? ((t.n + 63) / 64 + gy - 1) / gy : 0;
  const dim3 grid(t.nx + sums, gy);
  const size_t shm = std::max<size_t>(ConvTile<CIN>::lds(s.W, TP), 256 * sizeof(float));
  auto go = [&](auto k) {
    hipLaunchKernelGGL(k, grid, dim3(256), shm, c->stream, (const uint16_t*)in,
                       (const uint16_t*)wt, bias, (uint16_t*)out, out_f32, s, relu, t);
    return hipGetLastError();
  };
  constexpr int M = ConvTile<CIN>::CTMAX;
  if constexpr (M >= 4)
    if (ct == 4) return t.part ? go(k_conv3x3_tile<CIN, 4, TP, true>)
                               : go(k_conv3x3_tile<CIN, 4, TP, false>);
  if constexpr (M >= 2)
    if (ct == 2) return t.part ? go(k_conv3x3_tile<CIN, 2, TP, true>)
                               : go(k_conv3x3_tile<CIN, 2, TP, false>);
  return t.part ? go(k_conv3x3_tile<CIN, 1, TP, true>) : go(k_conv3x3_tile<CIN, 1, TP, false>);
}

// The tiled convolution where it applies (its channel counts, aligned tensors,
// staged rows within 96 KB): 256 pixels per block where that makes 256 blocks
// or more, else 64; as many output-channel tiles per block as leave 512
// blocks. Other shapes run k_conv3x3_fwd.
template <int CIN>
bool conv_tile(idmx_ctx_s* c, const void* in, const void* wt, const float* bias, void* out,
               float* out_f32, const ConvShape& s, int relu, const BwdWSum& t, hipError_t& e) {
  constexpr int M = ConvTile<CIN>::CTMAX;
  constexpr size_t LIM = 96 * 1024;
  const int P = s.N * s.H * s.W, cots = (s.Cout + 15) / 16;
  int ct = cots % 4 == 0 && M >= 4 ? 4 : cots % 2 == 0 && M >= 2 ? 2 : 1;
  const bool big = ConvTile<CIN>::lds(s.W, 256) <= LIM &&
                   (int64_t)(P + 255) / 256 * (cots / ct) >= 256;
  const int tp = big ? 256 : 64;
  if (ConvTile<CIN>::lds(s.W, tp) > LIM) return false;
  while (ct > 1 && (int64_t)(P + tp - 1) / tp * (cots / ct) < 512) ct /= 2;
  e = big ? conv_tile_ct<CIN, 256>(c, in, wt, bias, out, out_f32, s, relu, ct, t)
          : conv_tile_ct<CIN, 64>(c, in, wt, bias, out, out_f32, s, relu, ct, t);
  return true;
}

hipError_t launch_bwd_w_sum(idmx_ctx_s* c, const BwdWSum& t) {
  hipLaunchKernelGGL(k_conv_bwd_w_sum, dim3((t.n + 63) / 64), dim3(256), 0, c->stream, t);
  return hipGetLastError();
}

// With t.part the launch also adds up that weight gradient (a layer's
// backward-data pass).
hipError_t conv_fwd(idmx_ctx_s* c, const void* in, const void* wt, const float* bias, void* out,
                    float* out_f32, const ConvShape& s, int relu, const BwdWSum& t = {}) {
  hipError_t e = hipSuccess;
  if (aligned(in, 16) && aligned(wt, 8) && aligned(out, 8) && aligned(bias, 16) &&
      aligned(out_f32, 16)) {
    bool done = false;
    switch (s.Cin) {
      case 8: done = conv_tile<8>(c, in, wt, bias, out, out_f32, s, relu, t, e); break;
      case 16: done = conv_tile<16>(c, in, wt, bias, out, out_f32, s, relu, t, e); break;
      case 32: done = conv_tile<32>(c, in, wt, bias, out, out_f32, s, relu, t, e); break;
      case 64: done = conv_tile<64>(c, in, wt, bias, out, out_f32, s, relu, t, e); break;
      case 128: done = conv_tile<128>(c, in, wt, bias, out, out_f32, s, relu, t, e); break;
    }
    if (done) return e;
  }
  if (t.part) {
    e = launch_bwd_w_sum(c, t);
    if (e != hipSuccess) return e;
  }
  const int64_t waves = (int64_t)((s.N * s.H * s.W + 15) / 16) * ((s.Cout + 15) / 16);
  hipLaunchKernelGGL(k_conv3x3_fwd, dim3(g1(waves * 64)), dim3(256), 0, c->stream,
                     (const uint16_t*)in, (const uint16_t*)wt, bias, (uint16_t*)out, out_f32, s,
                     relu);
  return hipGetLastError();
}

// One layer's weight gradient: its operands, and with y the ReLU mask of dy
// (in place), with wd the backward-data weights from w, written by the same
// launch where the tiled kernels apply; with `later` the sums over the tiled
// kernel's parts are left to the caller's next launch (*later, before the
// parts are written again), which has nothing to do if later->part is null.
struct BwdWArgs {
  const void* in;
  void* dy;
  const void* y;
  float *dw, *db;
  const float* w;
  void* wd;
  BwdWSum* later = nullptr;
};

template <int CIN, int COUT, int TPX>
bool bwd_w_run(idmx_ctx_s* c, const BwdWArgs& a, const ConvShape& s, hipError_t& e) {
  using B = BwdW<CIN, COUT, TPX>;
  if (s.W % 4 || TPX % s.W || B::lds(s.W) > 160 * 1024) return false;
  const int P = s.N * s.H * s.W, nchunks = (P + TPX - 1) / TPX;
  const int blocks = std::min(nchunks, 256), nw = COUT * 9 * CIN;
  const size_t need = (size_t)blocks * (nw + COUT);
  if (need > c->nn_part_cap) {
    if (c->nn_part) {
      e = hipStreamSynchronize(c->stream);
      if (e == hipSuccess) e = hipFree(c->nn_part);
      if (e != hipSuccess) return true;
    }
    c->nn_part = nullptr;
    c->nn_part_cap = 0;
    e = hipMalloc(&c->nn_part, need * sizeof(float));
    if (e != hipSuccess) {  // no room: the kernel that needs no workspace
      (void)hipGetLastError();
      c->nn_part = nullptr;
      return false;
    }
    c->nn_part_cap = need;
  }
  const int flips = a.wd ? (nw + 255) / 256 : 0;
  hipLaunchKernelGGL((k_conv3x3_bwd_w_tile<CIN, COUT, TPX>), dim3(blocks + flips), dim3(256),
                     B::lds(s.W), c->stream, (const uint16_t*)a.in, (uint16_t*)a.dy,
                     (const uint16_t*)a.y, c->nn_part, s, nchunks, blocks, a.w, (uint16_t*)a.wd);
  e = hipGetLastError();
  if (e != hipSuccess) return true;
  BwdWSum t;
  t.part = c->nn_part;
  t.dw = a.dw;
  t.db = a.db;
  t.nw = nw;
  t.n = nw + COUT;
  t.parts = blocks;
  if (a.later) *a.later = t;
  else e = launch_bwd_w_sum(c, t);
  return true;
}

// Chunks of 256 pixels where they make 128 blocks, else of 64.
template <int CIN, int COUT>
bool bwd_w_tile(idmx_ctx_s* c, const BwdWArgs& a, const ConvShape& s, hipError_t& e) {
  const int P = s.N * s.H * s.W;
  if (P < 256 * 128 && bwd_w_run<CIN, COUT, 64>(c, a, s, e)) return true;
  return bwd_w_run<CIN, COUT, 256>(c, a, s, e);
}

template <int CIN>
bool bwd_w_cout(idmx_ctx_s* c, const BwdWArgs& a, const ConvShape& s, hipError_t& e) {
  switch (s.Cout) {
    case 1: return bwd_w_tile<CIN, 1>(c, a, s, e);
    case 16: return bwd_w_tile<CIN, 16>(c, a, s, e);
    case 32: return bwd_w_tile<CIN, 32>(c, a, s, e);
    case 64:
      if constexpr (CIN <= 64) return bwd_w_tile<CIN, 64>(c, a, s, e);
  }
  return false;
}

hipError_t relu_bwd(idmx_ctx_s* c, const void* y, const void* dy, void* dx, int64_t n) {
  if (n % 8 == 0 && aligned(y, 16) && aligned(dy, 16) && aligned(dx, 16))
    hipLaunchKernelGGL(k_relu_bwd8, dim3(g1(n / 8)), dim3(256), 0, c->stream, (const uint16_t*)y,
                       (const uint16_t*)dy, (uint16_t*)dx, n / 8);
  else
    hipLaunchKernelGGL(k_relu_bwd, dim3(g1(n)), dim3(256), 0, c->stream, (const uint16_t*)y,
                       (const uint16_t*)dy, (uint16_t*)dx, n);
  return hipGetLastError();
}

hipError_t flip_weights(idmx_ctx_s* c, const float* w, void* wd, int Cin, int Cout) {
  hipLaunchKernelGGL(k_conv_flip_weights, dim3(g1(Cin * 9 * Cout)), dim3(256), 0, c->stream, w,
                     (uint16_t*)wd, Cin, Cout);
  return hipGetLastError();
}

hipError_t bwd_weight(idmx_ctx_s* c, const BwdWArgs& a, const ConvShape& s) {
  hipError_t e = hipSuccess;
  // (no pixels, which idmx_nn_conv3x3_bwd_weight lets pass: nothing to add, and
  // nothing for the tiled kernels to divide by or to launch)
  const bool pixels = s.N > 0 && s.H > 0 && s.W > 0;
  if (pixels && aligned(a.in, 16) && aligned(a.dy, 16) && aligned(a.y, 16)) {
    bool done = false;
    switch (s.Cin) {
      case 8: done = bwd_w_cout<8>(c, a, s, e); break;
      case 16: done = bwd_w_cout<16>(c, a, s, e); break;
      case 32: done = bwd_w_cout<32>(c, a, s, e); break;
      case 64: done = bwd_w_cout<64>(c, a, s, e); break;
      case 128: done = bwd_w_cout<128>(c, a, s, e); break;
    }
    if (done) return e;
  }
  const int P = s.N * s.H * s.W;
  if (a.y) {
    e = relu_bwd(c, a.y, a.dy, a.dy, (int64_t)P * s.Cout);
    if (e != hipSuccess) return e;
  }
  const int pchunk = 1024;
  const int64_t waves = (int64_t)((s.Cout + 15) / 16) * ((9 * s.Cin + 15) / 16) *
                        ((P + pchunk - 1) / pchunk);
  hipLaunchKernelGGL(k_conv3x3_bwd_w, dim3(g1(waves * 64)), dim3(256), 0, c->stream,
                     (const uint16_t*)a.in, (const uint16_t*)a.dy, a.dw, s, pchunk);
  if (a.db)
    hipLaunchKernelGGL(k_bias_grad, dim3(s.Cout), dim3(256), 0, c->stream, (const uint16_t*)a.dy,
                       a.db, P, s.Cout);
  if (a.wd) return flip_weights(c, a.w, a.wd, s.Cin, s.Cout);
  return hipGetLastError();
}

}  // namespace idmx

using namespace idmx;

#define NCHECK(cond, msg)   \
  do {                      \
    if (!(cond)) {          \
      set_error(msg);       \
      return IDMX_E_ARG;    \
    }                       \
  } while (0)

extern "C" {

int idmx_nn_conv3x3_fwd(idmx_ctx_t c, const void* in, const void* wt, const float* bias,
                        void* out, float* out_f32, int N, int H, int W, int Cin, int Cout,
                        int relu) {
  NCHECK(c && in && wt && out && N > 0 && H > 0 && W > 0 && Cin > 0 && Cout > 0,
         "idmx_nn_conv3x3_fwd: invalid argument");
  IDMX_HIP(conv_fwd(c, in, wt, bias, out, out_f32, ConvShape{N, H, W, Cin, Cout}, relu));
  return IDMX_OK;
}

int idmx_nn_conv3x3_bwd_data(idmx_ctx_t c, const void* dy, const float* w, void* wd_scratch,
                             void* dx, int N, int H, int W, int Cin, int Cout) {
  NCHECK(c && dy && w && wd_scratch && dx && N > 0 && H > 0 && W > 0 && Cin > 0 && Cout > 0,
         "idmx_nn_conv3x3_bwd_data: invalid argument");
  IDMX_HIP(flip_weights(c, w, wd_scratch, Cin, Cout));
  IDMX_HIP(conv_fwd(c, dy, wd_scratch, nullptr, dx, nullptr, ConvShape{N, H, W, Cout, Cin}, 0));
  return IDMX_OK;
}

int idmx_nn_conv3x3_bwd_weight(idmx_ctx_t c, const void* in, const void* dy, float* dw,
                               float* db, int N, int H, int W, int Cin, int Cout) {
  NCHECK(c && in && dy && dw, "idmx_nn_conv3x3_bwd_weight: invalid argument");
  IDMX_HIP(bwd_weight(c, {in, (void*)dy, nullptr, dw, db, nullptr, nullptr},
                      ConvShape{N, H, W, Cin, Cout}));
  return IDMX_OK;
}

int idmx_nn_conv3x3_bwd(idmx_ctx_t c, const void* in, const void* y, void* dy, const float* w,
                        void* wd_scratch, void* dx, float* dw, float* db, int N, int H, int W,
                        int Cin, int Cout) {
  NCHECK(c && in && dy && w && dw && (!dx || wd_scratch) && N > 0 && H > 0 && W > 0 && Cin > 0 &&
             Cout > 0,
         "idmx_nn_conv3x3_bwd: invalid argument");
  BwdWSum t;
  IDMX_HIP(bwd_weight(c, {in, dy, y, dw, db, w, dx ? wd_scratch : nullptr, dx ? &t : nullptr},
                      ConvShape{N, H, W, Cin, Cout}));
  if (dx)
    IDMX_HIP(conv_fwd(c, dy, wd_scratch, nullptr, dx, nullptr, ConvShape{N, H, W, Cout, Cin}, 0,
                      t));
  return IDMX_OK;
}

int idmx_nn_relu_bwd(idmx_ctx_t c, const void* y, const void* dy, void* dx, int64_t n) {
  NCHECK(c && y && dy && dx && n >= 0, "idmx_nn_relu_bwd: invalid argument");
  IDMX_HIP(relu_bwd(c, y, dy, dx, n));
  return IDMX_OK;
}

int idmx_nn_pool2(idmx_ctx_t c, const void* x, void* y, int N, int H, int W, int C, int bwd) {
  NCHECK(c && x && y && H % 2 == 0 && W % 2 == 0, "idmx_nn_pool2: invalid argument");
  const int64_t tot = bwd ? (int64_t)N * H * W * C : (int64_t)N * (H / 2) * (W / 2) * C;
  if (!bwd && C % 8 == 0 && N * (H / 2) > 0 && aligned(x, 16) && aligned(y, 16))
    hipLaunchKernelGGL(k_pool2_fwd8, dim3(std::min(N * (H / 2), 65536)), dim3(256), 0, c->stream,
                       (const uint16_t*)x, (uint16_t*)y, N * (H / 2), W / 2, C / 8);
  else if (bwd)
    hipLaunchKernelGGL(k_pool2_bwd, dim3(g1(tot)), dim3(256), 0, c->stream, (const uint16_t*)x,
                       (uint16_t*)y, N, H, W, C);
  else
    hipLaunchKernelGGL(k_pool2_fwd, dim3(g1(tot)), dim3(256), 0, c->stream, (const uint16_t*)x,
                       (uint16_t*)y, N, H, W, C);
  IDMX_HIP(hipGetLastError());
  return IDMX_OK;
}

int idmx_nn_up2(idmx_ctx_t c, const void* x, void* y, int N, int H, int W, int C, int Cy, int c0,
                int bwd) {
  NCHECK(c && x && y && c0 >= 0 && c0 + C <= Cy, "idmx_nn_up2: invalid argument");
  const int64_t tot = bwd ? (int64_t)N * H * W * C : (int64_t)N * 4 * H * W * C;
  if (bwd && C % 8 == 0 && Cy % 8 == 0 && c0 % 8 == 0 && N * H > 0 && aligned(x, 16) &&
      aligned(y, 16))
    hipLaunchKernelGGL(k_up2_bwd8, dim3(std::min(N * H, 65536)), dim3(256), 0, c->stream,
                       (const uint16_t*)x, (uint16_t*)y, N * H, W, C / 8, Cy, c0);
  else if (bwd)
    hipLaunchKernelGGL(k_up2_bwd, dim3(g1(tot)), dim3(256), 0, c->stream, (const uint16_t*)x,
                       (uint16_t*)y, N, H, W, C, Cy, c0);
  else
    hipLaunchKernelGGL(k_up2_fwd, dim3(g1(tot)), dim3(256), 0, c->stream, (const uint16_t*)x,
                       (uint16_t*)y, N, H, W, C, Cy, c0);
  IDMX_HIP(hipGetLastError());
  return IDMX_OK;
}

int idmx_nn_copy_channels(idmx_ctx_t c, const void* x, void* y, int64_t P, int Cx, int cx0,
                          int Cy, int cy0, int C) {
  NCHECK(c && x && y && cx0 + C <= Cx && cy0 + C <= Cy, "idmx_nn_copy_channels: invalid argument");
  hipLaunchKernelGGL(k_copy_channels, dim3(g1(P * C)), dim3(256), 0, c->stream,
                     (const uint16_t*)x, (uint16_t*)y, P, Cx, cx0, Cy, cy0, C);
  IDMX_HIP(hipGetLastError());
  return IDMX_OK;
}

int idmx_nn_add(idmx_ctx_t c, const void* a, const void* b, void* y, int64_t n) {
  NCHECK(c && a && b && y, "idmx_nn_add: invalid argument");
  hipLaunchKernelGGL(k_add_bf16, dim3(g1(n)), dim3(256), 0, c->stream, (const uint16_t*)a,
                     (const uint16_t*)b, (uint16_t*)y, n);
  IDMX_HIP(hipGetLastError());
  return IDMX_OK;
}

int idmx_nn_cat_up2(idmx_ctx_t c, const void* x, const void* skip, void* y, int N, int H, int W,
                    int C, int Cs) {
  NCHECK(c && x && skip && y && N > 0 && H > 0 && W > 0 && C > 0 && Cs > 0,
         "idmx_nn_cat_up2: invalid argument");
  if (C % 8 == 0 && Cs % 8 == 0 && aligned(x, 16) && aligned(skip, 16) && aligned(y, 16)) {
    hipLaunchKernelGGL(k_cat_up2_8, dim3(std::min(N * 2 * H, 65536)), dim3(256), 0, c->stream,
                       (const uint16_t*)x, (const uint16_t*)skip, (uint16_t*)y, N * 2 * H, W,
                       C / 8, Cs / 8);
    IDMX_HIP(hipGetLastError());
    return IDMX_OK;
  }
  const int rc = idmx_nn_up2(c, x, y, N, H, W, C, C + Cs, 0, 0);
  return rc ? rc : idmx_nn_copy_channels(c, skip, y, (int64_t)N * 4 * H * W, Cs, 0, C + Cs, C, Cs);
}

int idmx_nn_pool2_bwd_add(idmx_ctx_t c, const void* dpool, const void* dcat, void* dx,
                          void* scratch, int N, int H, int W, int C, int Cc, int c0) {
  NCHECK(c && dpool && dcat && dx && scratch && N > 0 && H > 0 && W > 0 && H % 2 == 0 &&
             W % 2 == 0 && C > 0 && c0 >= 0 && c0 + C <= Cc,
         "idmx_nn_pool2_bwd_add: invalid argument");
  if (C % 8 == 0 && Cc % 8 == 0 && c0 % 8 == 0 && aligned(dpool, 16) && aligned(dcat, 16) &&
      aligned(dx, 16)) {
    hipLaunchKernelGGL(k_pool2_bwd_add8, dim3(std::min(N * H, 65536)), dim3(256), 0, c->stream,
                       (const uint16_t*)dpool, (const uint16_t*)dcat, (uint16_t*)dx, N * H, W,
                       C / 8, Cc, c0);
    IDMX_HIP(hipGetLastError());
    return IDMX_OK;
  }
  const int64_t P = (int64_t)N * H * W;
  int rc = idmx_nn_pool2(c, dpool, dx, N, H, W, C, 1);
  if (!rc) rc = idmx_nn_copy_channels(c, dcat, scratch, P, Cc, c0, C, 0, C);
  return rc ? rc : idmx_nn_add(c, dx, scratch, dx, P * C);
}

int idmx_nn_mse(idmx_ctx_t c, const float* pred, const float* tgt, void* grad, int64_t n,
                double* loss) {
  NCHECK(c && pred && tgt && grad && loss && n > 0, "idmx_nn_mse: invalid argument");
  const unsigned grid = std::min<unsigned>(g1(n), 1024);
  hipLaunchKernelGGL(k_mse, dim3(grid), dim3(256), 0, c->stream, pred, tgt, (uint16_t*)grad,
                     (float*)c->partials, n);
  IDMX_HIP(hipGetLastError());
  float h[1024];
  IDMX_HIP(hipMemcpyAsync(h, c->partials, sizeof(float) * grid, hipMemcpyDeviceToHost, c->stream));
  IDMX_HIP(hipStreamSynchronize(c->stream));
  double s = 0;
  for (unsigned k = 0; k < grid; k++) s += h[k];
  *loss = s;
  return IDMX_OK;
}

int idmx_nn_adam(idmx_ctx_t c, float* w, float* g, float* m, float* v, void* wb, int64_t n,
                 float lr, float b1, float b2, float eps, int t) {
  NCHECK(c && w && g && m && v && n > 0 && t >= 1, "idmx_nn_adam: invalid argument");
  const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
  hipLaunchKernelGGL(k_adam, dim3(g1(n)), dim3(256), 0, c->stream, w, g, m, v, (uint16_t*)wb, n,
                     lr, b1, b2, eps, c1, c2);
  IDMX_HIP(hipGetLastError());
  return IDMX_OK;
}

int idmx_nn_adam_set(idmx_ctx_t c, int count, float* const* w, float* const* g, float* const* m,
                     float* const* v, void* const* wb, const int64_t* n, float lr, float b1,
                     float b2, float eps, int t) {
  NCHECK(c && count > 0 && w && g && m && v && wb && n && t >= 1,
         "idmx_nn_adam_set: invalid argument");
  for (int k = 0; k < count; k++)
    NCHECK(w[k] && g[k] && m[k] && v[k] && n[k] > 0, "idmx_nn_adam_set: invalid argument");
  const float c1 = 1.f - powf(b1, (float)t), c2 = 1.f - powf(b2, (float)t);
  for (int k0 = 0; k0 < count; k0 += AdamSet::MAX) {
    AdamSet s{};
    s.count = std::min(count - k0, AdamSet::MAX);
    for (int k = 0; k < s.count; k++) {
      s.w[k] = w[k0 + k];
      s.g[k] = g[k0 + k];
      s.m[k] = m[k0 + k];
      s.v[k] = v[k0 + k];
      s.wb[k] = (uint16_t*)wb[k0 + k];
      s.n[k] = n[k0 + k];
      s.first[k + 1] = s.first[k] + (int)std::min<int64_t>((s.n[k] + 255) / 256, 1024);
    }
    hipLaunchKernelGGL(k_adam_set, dim3(s.first[s.count]), dim3(256), 0, c->stream, s, lr, b1, b2,
                       eps, c1, c2);
    IDMX_HIP(hipGetLastError());
  }
  return IDMX_OK;
}

int idmx_nn_cast(idmx_ctx_t c, const void* x, void* y, int64_t n, int to_bf16) {
  NCHECK(c && x && y && n >= 0, "idmx_nn_cast: invalid argument");
  if (to_bf16)
    hipLaunchKernelGGL(k_f32_to_bf16, dim3(g1(n)), dim3(256), 0, c->stream, (const float*)x,
                       (uint16_t*)y, n);
  else
    hipLaunchKernelGGL(k_bf16_to_f32, dim3(g1(n)), dim3(256), 0, c->stream, (const uint16_t*)x,
                       (float*)y, n);
  IDMX_HIP(hipGetLastError());
  return IDMX_OK;
}

int idmx_nn_resize_to_lattice(idmx_ctx_t c, const float* img, int S, double* n, int L,
                              double add) {
  NCHECK(c && img && n && S > 0 && L > 0, "idmx_nn_resize_to_lattice: invalid argument");
  hipLaunchKernelGGL(k_resize_to_lattice, dim3(g1((int64_t)L * L)), dim3(256), 0, c->stream, img,
                     S, n, L, add);
  IDMX_HIP(hipGetLastError());
  return IDMX_OK;
}

}  // extern "C"
