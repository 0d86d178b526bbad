// Learned Davidson preconditioner on gfx950: inference fused into the
// correction step, and the training kernels (forward, per-band loss
// coefficients, backward, ordered gradient reduction, Adam).
//
// One wave evaluates the network for 16 rows at a time. Lane l works on row
// e = l % 16 and on the hidden units 16*b + 4*(l/16) + i (b, i < 4): that is
// the B-operand layout of v_mfma_f32_16x16x16_bf16 for the 64 x 64 layer, and
// its D layout for the outputs, so h1 feeds the MFMA straight from registers
// and the layer-2 outputs land where the lane needs them. W2 is read as bf16
// from LDS; sums are FP32 (layers 1 and 3 on the VALU).
//
// Backward: delta2 (D layout) is the B operand of W2^T delta2; the weight
// gradient dW2 = sum_rows delta2 h1^T is an MFMA over the 16 rows of a group
// after a 16 x 16 transpose of delta2 and h1 through LDS. Gradients are
// accumulated per wave over a fixed set of groups and reduced in a fixed
// order, so a training step is bitwise deterministic.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <string>
#include <vector>

#include "common.hpp"
#include "mlp.hpp"

namespace bd {
namespace mlp {

namespace {
typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

// Blob header offsets (floats).
constexpr int hW1 = 0, hb1 = 256, hb2 = 320, hw3 = 384, hb3 = 448;

__device__ __forceinline__ unsigned short bf16_bits(float f) {
  unsigned int u = __float_as_uint(f);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return static_cast<unsigned short>(u >> 16);
}
__device__ __forceinline__ float bf16_value(float f) { return __uint_as_float(unsigned(bf16_bits(f)) << 16); }

// tanh(x) = 1 - 2 / (1 + e^{2x}) with the hardware reciprocal (1 ulp, no
// division sequence); saturates to +-1 for large |x| (rcp(inf) = 0).
__device__ __forceinline__ float tanh_f(float x) {
  return 1.0f - 2.0f * __builtin_amdgcn_rcpf(1.0f + __expf(2.0f * x));
}

__device__ __forceinline__ double wave_sum_d(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

struct Group {
  float h1[16];  // unit 16*kb + 4*q + i at [kb*4 + i]
  float h2[16];  // unit 16*rb + 4*q + i at [rb*4 + i]
  bf16x4 hb[4];  // bf16(h1), the MFMA B operand
  float o;       // network output of the lane's row (same in all four quads)
};

// W2 (and W2^T) rows in LDS, 4 bf16 of padding each: the 16 rows an A-operand
// read touches then start in different banks (64-element rows all start in
// two).
constexpr int kRowW2 = kHidden + 4;
constexpr int kLdsW2 = 512, kLdsW2T = kLdsW2 + kHidden * kRowW2 / 2, kLdsFloats = kLdsW2T + kHidden * kRowW2 / 2;

// LDS traffic between the lanes of one wave: its LDS instructions complete in
// order, so only the compiler has to be held back.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Network output for the lane's row from features u (sb: the blob in LDS).
__device__ __forceinline__ void forward_group(const float* sb, float u0, float u1, float u2, float u3, Group& G) {
  const int lane = threadIdx.x & 63, q = lane >> 4, e = lane & 15;
  const unsigned short* W2 = reinterpret_cast<const unsigned short*>(sb + kLdsW2);
#pragma unroll
  for (int kb = 0; kb < 4; ++kb)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 16 * kb + 4 * q + i;
      const float z = fmaf(sb[hW1 + 4 * n], u0,
                           fmaf(sb[hW1 + 4 * n + 1], u1, fmaf(sb[hW1 + 4 * n + 2], u2,
                                                              fmaf(sb[hW1 + 4 * n + 3], u3, sb[hb1 + n]))));
      const float h = tanh_f(z);
      G.h1[kb * 4 + i] = h;
      G.hb[kb][i] = static_cast<short>(bf16_bits(h));
    }
  float part = 0.0f;
#pragma unroll
  for (int rb = 0; rb < 4; ++rb) {
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < 4; ++kb) {
      const bf16x4 a = *reinterpret_cast<const bf16x4*>(&W2[(16 * rb + e) * kRowW2 + 16 * kb + 4 * q]);
      acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, G.hb[kb], acc, 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = 16 * rb + 4 * q + i;
      const float h2 = tanh_f(acc[i] + sb[hb2 + n]);
      G.h2[rb * 4 + i] = h2;
      part = fmaf(sb[hw3 + n], h2, part);
    }
  }
  part += __shfl_xor(part, 16, 64);
  part += __shfl_xor(part, 32, 64);
  G.o = part + sb[hb3];
}

// The blob into LDS: inference reads W1, the biases, w3 and W2 (the first
// kLdsW2T floats); training also reads W2^T.
template <bool train>
__device__ __forceinline__ void load_blob(float* sb, const float* blob) {
  constexpr int half = kHidden / 2, count = train ? kBlobFloats : kBlobW2T;
  for (int i = threadIdx.x; i < count; i += blockDim.x) {
    int at = i;
    if (i >= kBlobW2) {
      const int r = (i - kBlobW2) / half;  // (W2^T's rows follow W2's)
      at = kLdsW2 + r * (kRowW2 / 2) + (i - kBlobW2) % half;
    }
    sb[at] = blob[i];
  }
  __syncthreads();
}

__device__ __forceinline__ float band_u1(float T) { return logf(T); }

// ---------------------------------------------------------------------------
// Parameters -> inference blob.
// ---------------------------------------------------------------------------
__global__ void k_quantize(const float* __restrict__ th, float* __restrict__ blob) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  unsigned short* W2 = reinterpret_cast<unsigned short*>(blob + kBlobW2);
  unsigned short* W2T = reinterpret_cast<unsigned short*>(blob + kBlobW2T);
  if (t < kHidden * kHidden) {
    const int out = t / kHidden, in = t % kHidden;
    const unsigned short b = bf16_bits(th[oW2 + t]);
    W2[out * kHidden + in] = b;
    W2T[in * kHidden + out] = b;
  }
  if (t < 512) {
    float v = 0.0f;
    if (t < 256) v = bf16_value(th[oW1 + t]);
    else if (t < 320) v = th[ob1 + t - 256];
    else if (t < 384) v = th[ob2 + t - 320];
    else if (t < 448) v = bf16_value(th[ow3 + t - 384]);
    else if (t == 448) v = th[ob3];
    blob[t] = v;
  }
}

// ---------------------------------------------------------------------------
// Inference inside the Davidson correction step.
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(256) void k_kinetic_scale(const double* __restrict__ X, int64_t n,
                                                       const double* __restrict__ kinetic, double* __restrict__ T) {
  __shared__ double red[2][4];
  const int j = blockIdx.x;
  const double* x = X + int64_t(j) * n;
  double a = 0.0, b = 0.0;
  const int64_t S = blockDim.x;
  int64_t i = threadIdx.x;
  // Four rows a pass with their loads issued first; the sums run in row
  // order, as in the one-row loop below.
  for (; i + 3 * S < n; i += 4 * S) {
    double xv[4], kv[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      xv[u] = x[i + u * S];
      kv[u] = kinetic[i + u * S];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const double w = xv[u] * xv[u];
      a += w * kv[u];
      b += w;
    }
  }
  for (; i < n; i += S) {
    const double w = x[i] * x[i];
    a += w * kinetic[i];
    b += w;
  }
  a = wave_sum_d(a);
  b = wave_sum_d(b);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    red[0][wave] = a;
    red[1][wave] = b;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    const double sa = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    const double sb = red[1][0] + red[1][1] + red[1][2] + red[1][3];
    T[j] = fmax(sa / sb, double(kKineticFloor));
  }
}

__global__ __launch_bounds__(256) void k_correct(int64_t n, const double* __restrict__ X, const double* __restrict__ HX,
                                                 const double* __restrict__ theta_ritz, const double* __restrict__ Tb,
                                                 const double* __restrict__ kinetic,
                                                 const double* __restrict__ diag, double vbar,
                                                 const float* __restrict__ blob, double* __restrict__ E,
                                                 double* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) float sb[kLdsW2T];
  __shared__ double red[2][4];
  load_blob<false>(sb, blob);
  const int j = blockIdx.y, lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4, e = lane & 15;
  const double th = theta_ritz[j];
  const float T = float(Tb[j]);
  const float u1 = band_u1(T), u2 = float((th - vbar) / Tb[j]), u3 = float(vbar);
  const double* x = X + int64_t(j) * n;
  const double* hx = HX + int64_t(j) * n;
  double* ej = E + int64_t(j) * n;
  double se = 0.0, sr = 0.0;
  const int64_t stride = int64_t(gridDim.x) * 64;
  int64_t row = int64_t(blockIdx.x) * 64 + 16 * wave + e;
  float g_next = row < n ? float(kinetic[row]) : 0.0f;
  for (int64_t base = int64_t(blockIdx.x) * 64; base < n; base += stride, row += stride) {
    const bool ok = row < n;
    const float g = g_next;
    // This pass's operands and the next pass's row energy are loaded before
    // the network runs, so their latency hides behind it.
    double xr = 0.0, hr = 0.0, dr = 0.0;
    if (ok && q == 0) {
      xr = x[row];
      hr = hx[row];
      dr = diag[row];
    }
    const int64_t next = row + stride;
    g_next = next < n ? float(kinetic[next]) : 0.0f;
    Group G;
    forward_group(sb, log1pf(g / T), u1, u2, u3, G);
    if (ok && q == 0) {
      const double r = hr - th * xr;
      const double v = -double(expf(G.o)) * r / qe_denominator(dr, th);
      ej[row] = v;
      se += v * v;
      sr += r * r;
    }
  }
  se = wave_sum_d(se);
  sr = wave_sum_d(sr);
  if (lane == 0) {
    red[0][wave] = se;
    red[1][wave] = sr;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    double* p = part + (int64_t(j) * gridDim.x + blockIdx.x) * 2;
    p[0] = red[0][0] + red[0][1] + red[0][2] + red[0][3];
    p[1] = red[1][0] + red[1][1] + red[1][2] + red[1][3];
  }
}

__global__ void k_reduce_norms(int k, int nblk, const double* __restrict__ part, double* __restrict__ n2e,
                               double* __restrict__ n2r) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j >= k) return;
  double a = 0.0, b = 0.0;
  for (int p = 0; p < nblk; ++p) {
    a += part[(int64_t(j) * nblk + p) * 2];
    b += part[(int64_t(j) * nblk + p) * 2 + 1];
  }
  n2e[j] = a;
  n2r[j] = b;
}

__global__ __launch_bounds__(256) void k_forward_k(int64_t n, const float* __restrict__ g, float T, float ritz,
                                                   float vbar, const float* __restrict__ blob, float* __restrict__ K) {
  __shared__ __attribute__((aligned(16))) float sb[kLdsW2T];
  load_blob<false>(sb, blob);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4, e = lane & 15;
  const float u1 = band_u1(T), u2 = (ritz - vbar) / T, u3 = vbar;
  for (int64_t base = int64_t(blockIdx.x) * 64; base < n; base += int64_t(gridDim.x) * 64) {
    const int64_t row = base + 16 * wave + e;
    const bool ok = row < n;
    Group G;
    forward_group(sb, log1pf((ok ? g[row] : 0.0f) / T), u1, u2, u3, G);
    if (ok && q == 0) K[row] = expf(G.o);
  }
}

// ---------------------------------------------------------------------------
// Training.
// ---------------------------------------------------------------------------
struct BandIn {
  float u1, u2, u3, T;
};
__device__ __forceinline__ BandIn band_in(const float* scal, int b) {
  BandIn B;
  B.T = scal[3 * b];
  B.u1 = band_u1(B.T);
  B.u2 = (scal[3 * b + 1] - scal[3 * b + 2]) / B.T;
  B.u3 = scal[3 * b + 2];
  return B;
}

// Per band of the batch and block: sum a t, sum a a, sum t t (a = K r).
__global__ __launch_bounds__(256) void k_train_fwd(TrainSet ts, const int* __restrict__ batch,
                                                   const float* __restrict__ blob, double* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) float sb[kLdsW2T];
  __shared__ double red[3][4];
  load_blob<false>(sb, blob);
  const int bi = blockIdx.y, b = batch[bi];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4, e = lane & 15;
  const BandIn B = band_in(ts.scal, b);
  const float* R = ts.R + int64_t(b) * ts.n;
  const float* Tg = ts.Tg + int64_t(b) * ts.n;
  double c = 0.0, aa = 0.0, tt = 0.0;
  for (int64_t base = int64_t(blockIdx.x) * 64; base < ts.n; base += int64_t(gridDim.x) * 64) {
    const int64_t row = base + 16 * wave + e;
    const bool ok = row < ts.n;
    Group G;
    forward_group(sb, log1pf((ok ? ts.g[row] : 0.0f) / B.T), B.u1, B.u2, B.u3, G);
    if (ok && q == 0) {
      const double a = double(expf(G.o)) * double(R[row]);
      const double t = Tg[row];
      c += a * t;
      aa += a * a;
      tt += t * t;
    }
  }
  c = wave_sum_d(c);
  aa = wave_sum_d(aa);
  tt = wave_sum_d(tt);
  if (lane == 0) {
    red[0][wave] = c;
    red[1][wave] = aa;
    red[2][wave] = tt;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const int s = threadIdx.x;
    part[(int64_t(bi) * gridDim.x + blockIdx.x) * 3 + s] = red[s][0] + red[s][1] + red[s][2] + red[s][3];
  }
}

// Loss and dL/da = alpha t + beta a per batch band (mean over the batch): a
// wave per band, then the bands in order. (One thread over all of it spent 115
// us on 16 bands of 64 blocks, a load's latency each.)
__global__ __launch_bounds__(256) void k_band_coef(int batch, int nblk, const double* __restrict__ part,
                                                   double* __restrict__ coef, double* __restrict__ loss) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  __shared__ double band_loss[4];
  double total = 0.0;
  for (int b0 = 0; b0 < batch; b0 += 4) {
    const int bi = b0 + wave;
    if (bi < batch) {
      double c = 0.0, A = 0.0, B = 0.0;
      for (int p = lane; p < nblk; p += 64) {
        c += part[(int64_t(bi) * nblk + p) * 3];
        A += part[(int64_t(bi) * nblk + p) * 3 + 1];
        B += part[(int64_t(bi) * nblk + p) * 3 + 2];
      }
      c = wave_sum_d(c);
      A = wave_sum_d(A);
      B = wave_sum_d(B);
      if (lane == 0) {
        double L = 1.0, alpha = 0.0, beta = 0.0;
        if (A > 0.0 && B > 0.0) {
          L = 1.0 - c * c / (A * B);
          alpha = -2.0 * c / (A * B) / batch;
          beta = 2.0 * c * c / (A * A * B) / batch;
        }
        coef[2 * bi] = alpha;
        coef[2 * bi + 1] = beta;
        band_loss[wave] = L;
      }
    }
    __syncthreads();
    if (threadIdx.x == 0)
      for (int w = 0; w < 4 && b0 + w < batch; ++w) total += band_loss[w];
    __syncthreads();
  }
  if (threadIdx.x == 0) loss[0] = total / batch;
}

// Backward over all rows of the batch; per-workgroup gradient partials (kCount
// floats each, the four waves added in order). A wave's groups follow one
// another and its LDS transposes are its own: no barrier in the loop.
// Bound by the transcendentals of the tanh (two a unit and row) and by the
// VALU, so the chip needs every SIMD: about 512 workgroups (two waves a SIMD,
// what the registers allow). 16 bands of 23,847 rows: 317 -> 94 us (128
// workgroups before, with the weight rows in two banks and a barrier twice a
// group).
__global__ __launch_bounds__(256, 2) void k_train_bwd(TrainSet ts, const int* __restrict__ batch, int nbatch,
                                                   const float* __restrict__ blob, const double* __restrict__ coef,
                                                   float* __restrict__ part) {
  __shared__ __attribute__((aligned(16))) float sb[kLdsFloats];
  __shared__ __attribute__((aligned(16))) unsigned short d2T[4][64 * 16];  // per wave: delta2[unit][row]
  __shared__ __attribute__((aligned(16))) unsigned short h1T[4][64 * 16];  // per wave: bf16(h1)[unit][row]
  load_blob<true>(sb, blob);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, q = lane >> 4, e = lane & 15;
  const unsigned short* W2T = reinterpret_cast<const unsigned short*>(sb + kLdsW2T);
  const int64_t gpb = (ts.n + 15) / 16;  // row groups per band
  const int64_t total = gpb * nbatch, waves = int64_t(gridDim.x) * 4;
  const int64_t per = (total + waves - 1) / waves;  // groups of a wave, one after the other
  const int64_t first = (int64_t(blockIdx.x) * 4 + wave) * per, last = min(first + per, total);
  f32x4 dW2[4][4];
#pragma unroll
  for (int a = 0; a < 4; ++a)
#pragma unroll
    for (int c = 0; c < 4; ++c) dW2[a][c] = f32x4{0.f, 0.f, 0.f, 0.f};
  float dW1[16], db1[16], db2[16], dw3[16], db3 = 0.0f;
#pragma unroll
  for (int k = 0; k < 16; ++k) dW1[k] = db1[k] = db2[k] = dw3[k] = 0.0f;
  // Features 1 to 3 are the band's, the same in all its rows: a band's sum of
  // delta1 gives their gradients, folded in when the wave leaves the band.
  __shared__ float folded[4][kHidden][4];  // per wave and unit: db1, dW1[1 .. 3]
#pragma unroll
  for (int i = 0; i < 4; ++i) folded[wave][lane][i] = 0.0f;
  wave_sync();
  auto sum_rows = [](float v) {  // over the 16 rows held by lanes of the same quad
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) v += __shfl_xor(v, off, 64);
    return v;
  };
  auto fold = [&](const BandIn& B) {
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      const float v = sum_rows(db1[k]);
      db1[k] = 0.0f;
      if (e == 0) {
        float* f = folded[wave][16 * (k >> 2) + 4 * q + (k & 3)];
        f[0] += v;
        f[1] = fmaf(v, B.u1, f[1]);
        f[2] = fmaf(v, B.u2, f[2]);
        f[3] = fmaf(v, B.u3, f[3]);
      }
    }
  };
  int bi = int(min(first, total - 1) / gpb);
  int64_t group = first - bi * gpb;  // within band bi
  int b = batch[bi];
  BandIn B = band_in(ts.scal, b);
  // The next group's row is loaded while this one runs through the network.
  float g_next = 0.0f, r_next = 0.0f, t_next = 0.0f;
  auto fetch = [&](int64_t row, int band) {
    const int64_t at = min(row, ts.n - 1);
    g_next = ts.g[at];
    r_next = ts.R[int64_t(band) * ts.n + at];
    t_next = ts.Tg[int64_t(band) * ts.n + at];
  };
  if (first < last) fetch(group * 16 + e, b);
  for (int64_t done = first; done < last; ++done, ++group) {
    if (group >= gpb) {
      fold(B);
      group = 0;
      b = batch[++bi];
      B = band_in(ts.scal, b);
    }
    const bool ok = group * 16 + e < ts.n;
    const float g = g_next, r = r_next, t = t_next;
    if (done + 1 < last) {
      if (group + 1 < gpb) fetch((group + 1) * 16 + e, b);
      else fetch(e, batch[bi + 1]);
    }
    const float u0 = log1pf((ok ? g : 0.0f) / B.T);
    Group G;
    forward_group(sb, u0, B.u1, B.u2, B.u3, G);
    float dLdo = 0.0f;
    if (ok) {
      const float K = expf(G.o);
      const double a = double(K) * double(r);
      dLdo = float((coef[2 * bi] * t + coef[2 * bi + 1] * a) * double(r) * double(K));
    }
    if (q == 0) db3 += dLdo;
    bf16x4 d2b[4];
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = 16 * rb + 4 * q + i;
        const float h2 = G.h2[rb * 4 + i];
        dw3[rb * 4 + i] = fmaf(dLdo, h2, dw3[rb * 4 + i]);
        const float d2 = dLdo * sb[hw3 + n] * (1.0f - h2 * h2);
        db2[rb * 4 + i] += d2;
        const unsigned short bits = bf16_bits(d2);
        d2b[rb][i] = static_cast<short>(bits);
        d2T[wave][n * 16 + e] = bits;
      }
    // delta1 = (W2^T delta2) * (1 - h1^2).
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kb = 0; kb < 4; ++kb) {
        const bf16x4 a = *reinterpret_cast<const bf16x4*>(&W2T[(16 * rb + e) * kRowW2 + 16 * kb + 4 * q]);
        acc = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, d2b[kb], acc, 0, 0, 0);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int k = rb * 4 + i;
        const float h1 = G.h1[k];
        const float d1 = acc[i] * (1.0f - h1 * h1);
        db1[k] += d1;
        dW1[k] = fmaf(d1, u0, dW1[k]);
        h1T[wave][(16 * rb + 4 * q + i) * 16 + e] = static_cast<unsigned short>(G.hb[rb][i]);
      }
    }
    wave_sync();
    // dW2[out][in] += sum_rows delta2[out][row] h1[in][row].
#pragma unroll
    for (int rb = 0; rb < 4; ++rb) {
      const bf16x4 a = *reinterpret_cast<const bf16x4*>(&d2T[wave][(16 * rb + e) * 16 + 4 * q]);
#pragma unroll
      for (int cb = 0; cb < 4; ++cb) {
        const bf16x4 bb = *reinterpret_cast<const bf16x4*>(&h1T[wave][(16 * cb + e) * 16 + 4 * q]);
        dW2[rb][cb] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, bb, dW2[rb][cb], 0, 0, 0);
      }
    }
    wave_sync();
  }
  fold(B);
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    dW1[k] = sum_rows(dW1[k]);
    db2[k] = sum_rows(db2[k]);
    dw3[k] = sum_rows(dw3[k]);
  }
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) db3 += __shfl_xor(db3, off, 64);
  // The waves add their gradients one after the other, over the blob.
  static_assert(kCount <= kLdsFloats, "gradient over the blob");
  float* P = sb;
  for (int w = 0; w < 4; ++w) {
    __syncthreads();
    if (wave != w) continue;
    auto put = [&](int at, float v) { P[at] = w == 0 ? v : P[at] + v; };
#pragma unroll
    for (int rb = 0; rb < 4; ++rb)
#pragma unroll
      for (int cb = 0; cb < 4; ++cb)
#pragma unroll
        for (int i = 0; i < 4; ++i) put(oW2 + (16 * rb + 4 * q + i) * kHidden + 16 * cb + e, dW2[rb][cb][i]);
    if (e == 0) {
#pragma unroll
      for (int b4 = 0; b4 < 4; ++b4)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = b4 * 4 + i, n = 16 * b4 + 4 * q + i;
          const float* f = folded[wave][n];
          put(oW1 + 4 * n, dW1[k]);
          put(oW1 + 4 * n + 1, f[1]);
          put(oW1 + 4 * n + 2, f[2]);
          put(oW1 + 4 * n + 3, f[3]);
          put(ob1 + n, f[0]);
          put(ob2 + n, db2[k]);
          put(ow3 + n, dw3[k]);
        }
    }
    if (lane == 0) put(ob3, db3);
  }
  __syncthreads();
  for (int i = threadIdx.x; i < kCount; i += 256) part[int64_t(blockIdx.x) * kCount + i] = P[i];
}

// Sum of the workgroups' partials in a fixed order: 16 segments of them side
// by side (a load's latency a partial bound the one-thread sums: 127 us for
// 512 partials), then the segments in order.
constexpr int kReduceSeg = 16;
__global__ __launch_bounds__(64 * kReduceSeg) void k_grad_reduce(int parts, const float* __restrict__ part,
                                                                 float* __restrict__ grad) {
  __shared__ double sum[kReduceSeg][64];
  const int lane = threadIdx.x & 63, seg = threadIdx.x >> 6;
  const int p = blockIdx.x * 64 + lane;
  const int per = (parts + kReduceSeg - 1) / kReduceSeg, end = min(parts, (seg + 1) * per);
  double s = 0.0;
  if (p < kCount) {
    int w = seg * per;
    for (; w + 8 <= end; w += 8) {
      float v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = part[int64_t(w + u) * kCount + p];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; w < end; ++w) s += part[int64_t(w) * kCount + p];
  }
  sum[seg][lane] = s;
  __syncthreads();
  if (seg != 0 || p >= kCount) return;
  s = 0.0;
#pragma unroll
  for (int g = 0; g < kReduceSeg; ++g) s += sum[g][lane];
  grad[p] = float(s);
}

__global__ void k_adam(float* __restrict__ th, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, float c1, float c2, float lr) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= kCount) return;
  const float b1 = 0.9f, b2 = 0.999f;
  const float mm = b1 * m[p] + (1.0f - b1) * g[p];
  const float vv = b2 * v[p] + (1.0f - b2) * g[p] * g[p];
  m[p] = mm;
  v[p] = vv;
  th[p] -= lr * (mm / c1) / (sqrtf(vv / c2) + 1e-8f);
}

constexpr int kCorrectBlocks = 128;
constexpr int kTrainFwdBlocks = 64;
constexpr int kTrainBwdBlocks = 512;

// Workgroups of the backward kernel: at least four groups a wave, so that a
// small batch does not spend its time on partial gradients.
int bwd_blocks(int64_t n, int batch) {
  return int(std::max<int64_t>(1, std::min<int64_t>(kTrainBwdBlocks, (n + 15) / 16 * batch / 16)));
}
}  // namespace

void quantize(hipStream_t s, const float* theta, float* blob) {
  hipLaunchKernelGGL(k_quantize, dim3((kHidden * kHidden + 255) / 256), dim3(256), 0, s, theta, blob);
}

int64_t correct_work(int64_t n, int k) {
  const int64_t nblk = std::min<int64_t>((n + 63) / 64, kCorrectBlocks);
  return k + 2 * int64_t(k) * nblk;
}

void correct(hipStream_t s, int64_t n, int k, const double* X, const double* HX, const double* theta_ritz,
             const double* kinetic, const double* diag, double vbar, const float* blob, double* E,
             double* norm2_e, double* norm2_r, double* work) {
  if (k <= 0) return;
  // About 4096 workgroups in all (each loads the network once), at most
  // kCorrectBlocks per column and at least 16.
  const int per_column = std::min(kCorrectBlocks, std::max(16, 4096 / k));
  const int nblk = int(std::min<int64_t>((n + 63) / 64, per_column));
  double* Tb = work;
  double* part = work + k;
  hipLaunchKernelGGL(k_kinetic_scale, dim3(k), dim3(256), 0, s, X, n, kinetic, Tb);
  hipLaunchKernelGGL(k_correct, dim3(nblk, k), dim3(256), 0, s, n, X, HX, theta_ritz, Tb, kinetic, diag, vbar, blob,
                     E, part);
  hipLaunchKernelGGL(k_reduce_norms, dim3((k + 63) / 64), dim3(64), 0, s, k, nblk, part, norm2_e, norm2_r);
}

int64_t train_work(int64_t n, int batch) {
  // fwd partials, coefficients, loss, then float gradient partials (as doubles).
  const int64_t fwd = 3 * int64_t(batch) * kTrainFwdBlocks;
  const int64_t bwd = (int64_t(bwd_blocks(n, batch)) * kCount + 1) / 2;
  return fwd + 2 * int64_t(batch) + 2 + bwd + 1;  // + the loss word
}

void loss_grad(hipStream_t s, const TrainSet& ts, const int* batch_dev, int batch, const float* blob, float* grad,
               double* loss, double* work) {
  if (batch <= 0 || ts.n <= 0) fail(BD_ERR_INVALID_PARAMETER, "empty training batch");
  double* fwd = work;
  double* coef = fwd + 3 * int64_t(batch) * kTrainFwdBlocks;
  float* gpart = reinterpret_cast<float*>(coef + 2 * int64_t(batch) + 2);
  hipLaunchKernelGGL(k_train_fwd, dim3(kTrainFwdBlocks, batch), dim3(256), 0, s, ts, batch_dev, blob, fwd);
  hipLaunchKernelGGL(k_band_coef, dim3(1), dim3(256), 0, s, batch, kTrainFwdBlocks, fwd, coef, loss);
  const int blocks = bwd_blocks(ts.n, batch);
  hipLaunchKernelGGL(k_train_bwd, dim3(blocks), dim3(256), 0, s, ts, batch_dev, batch, blob, coef, gpart);
  hipLaunchKernelGGL(k_grad_reduce, dim3((kCount + 63) / 64), dim3(64 * kReduceSeg), 0, s, blocks, gpart, grad);
}

void adam(hipStream_t s, float* theta, const float* grad, float* m, float* v, int step, float lr) {
  const float c1 = 1.0f - powf(0.9f, float(step));
  const float c2 = 1.0f - powf(0.999f, float(step));
  hipLaunchKernelGGL(k_adam, dim3((kCount + 255) / 256), dim3(256), 0, s, theta, grad, m, v, c1, c2, lr);
}

void forward_k(hipStream_t s, int64_t n, const float* g, float T, float theta_ritz, float vbar, const float* blob,
               float* K) {
  const int nblk = int(std::min<int64_t>((n + 63) / 64, 1024));
  hipLaunchKernelGGL(k_forward_k, dim3(nblk), dim3(256), 0, s, n, g, T, theta_ritz, vbar, blob, K);
}

}  // namespace mlp
}  // namespace bd

// ---------------------------------------------------------------------------
// C ABI.
// ---------------------------------------------------------------------------
namespace {
bd::mlp::TrainSet train_set(int64_t n, int32_t bands, const float* g, const float* R, const float* Tg,
                            const float* scal) {
  if (n <= 0 || bands <= 0 || !g || !R || !Tg || !scal) bd::fail(BD_ERR_INVALID_PARAMETER, "training set");
  bd::mlp::TrainSet ts;
  ts.n = n;
  ts.bands = bands;
  ts.g = g;
  ts.R = R;
  ts.Tg = Tg;
  ts.scal = scal;
  return ts;
}
void device_check(const char* what) {
  if (hipDeviceSynchronize() != hipSuccess || hipGetLastError() != hipSuccess)
    bd::fail(BD_ERR_DEVICE, std::string(what) + " failed on the device");
}
}  // namespace

extern "C" int32_t bd_mlp_param_count(void) { return bd::mlp::kCount; }
extern "C" int32_t bd_mlp_blob_floats(void) { return bd::mlp::kBlobFloats; }

extern "C" bd_status bd_mlp_quantize_dev(const float* theta, float* blob) {
  BD_GUARD({
    if (!theta || !blob) bd::fail(BD_ERR_INVALID_PARAMETER, "null argument");
    bd::mlp::quantize(nullptr, theta, blob);
    device_check("bd_mlp_quantize_dev");
  });
}

extern "C" bd_status bd_mlp_forward_dev(int64_t n, const float* g, float T, float ritz, float vbar, const float* blob,
                                        float* K) {
  BD_GUARD({
    if (n <= 0 || !g || !blob || !K || !(T > 0.0f)) bd::fail(BD_ERR_INVALID_PARAMETER, "mlp forward arguments");
    bd::mlp::forward_k(nullptr, n, g, T, ritz, vbar, blob, K);
    device_check("bd_mlp_forward_dev");
  });
}

extern "C" int64_t bd_mlp_train_workspace(int64_t n, int32_t batch) {
  return batch > 0 ? bd::mlp::train_work(n, batch) : 0;
}

extern "C" bd_status bd_mlp_loss_grad_dev(int64_t n, int32_t bands, const float* g, const float* R, const float* Tg,
                                          const float* scal, const int32_t* batch_dev, int32_t batch,
                                          const float* blob, float* grad, double* loss, double* work) {
  BD_GUARD({
    const bd::mlp::TrainSet ts = train_set(n, bands, g, R, Tg, scal);
    if (!batch_dev || batch <= 0 || !blob || !grad || !loss || !work)
      bd::fail(BD_ERR_INVALID_PARAMETER, "mlp loss arguments");
    double* dloss = work + bd::mlp::train_work(n, batch) - 1;
    bd::mlp::loss_grad(nullptr, ts, batch_dev, batch, blob, grad, dloss, work);
    if (hipMemcpy(loss, dloss, sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
      bd::fail(BD_ERR_DEVICE, "mlp loss readback");
    device_check("bd_mlp_loss_grad_dev");
  });
}

extern "C" bd_status bd_mlp_adam_dev(float* theta, const float* grad, float* m, float* v, int32_t step, float lr) {
  BD_GUARD({
    if (!theta || !grad || !m || !v || step < 1) bd::fail(BD_ERR_INVALID_PARAMETER, "adam arguments");
    bd::mlp::adam(nullptr, theta, grad, m, v, step, lr);
    device_check("bd_mlp_adam_dev");
  });
}

extern "C" bd_status bd_mlp_train_dev(int64_t n, int32_t bands, const float* g, const float* R, const float* Tg,
                                      const float* scal, float* theta, float* m, float* v, int32_t steps,
                                      int32_t batch, float lr, uint64_t seed, double* losses, int32_t* batch_dev,
                                      float* blob, float* grad, double* work) {
  BD_GUARD({
    const bd::mlp::TrainSet ts = train_set(n, bands, g, R, Tg, scal);
    if (!theta || !m || !v || steps < 0 || batch <= 0 || batch > bands || !losses || !batch_dev || !blob || !grad ||
        !work)
      bd::fail(BD_ERR_INVALID_PARAMETER, "mlp training arguments");
    double* dloss = work + bd::mlp::train_work(n, batch) - 1;
    std::vector<int32_t> idx(batch);
    uint64_t state = seed * 6364136223846793005ull + 1442695040888963407ull;
    for (int step = 1; step <= steps; ++step) {
      // Partial Fisher-Yates draw of `batch` distinct bands (64-bit LCG).
      std::vector<int32_t> pool(bands);
      for (int i = 0; i < bands; ++i) pool[i] = i;
      for (int i = 0; i < batch; ++i) {
        state = state * 6364136223846793005ull + 1442695040888963407ull;
        const int j = i + int((state >> 33) % uint64_t(bands - i));
        std::swap(pool[i], pool[j]);
        idx[i] = pool[i];
      }
      if (hipMemcpy(batch_dev, idx.data(), sizeof(int32_t) * batch, hipMemcpyHostToDevice) != hipSuccess)
        bd::fail(BD_ERR_DEVICE, "batch upload");
      bd::mlp::quantize(nullptr, theta, blob);
      bd::mlp::loss_grad(nullptr, ts, batch_dev, batch, blob, grad, dloss, work);
      bd::mlp::adam(nullptr, theta, grad, m, v, step, lr);
      if (hipMemcpy(&losses[step - 1], dloss, sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
        bd::fail(BD_ERR_DEVICE, "loss readback");
    }
    bd::mlp::quantize(nullptr, theta, blob);
    device_check("bd_mlp_train_dev");
  });
}
