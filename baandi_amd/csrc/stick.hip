// The x pass. A wavefront owns whole sticks: `per` lines of n0 = A B
// points, pass one as A-point transforms (B of them a line, one per lane),
// pass two as B-point transforms, the values changing lanes in the line's own
// LDS row, which only this wavefront touches. The inverse reads the ORC
// columns straight into the lanes that transform them (a table names each
// lane's representatives; most of a stick is outside the sphere) and writes the
// stick buffer from registers; the forward pass reads it the same way and
// crosses the workgroup once, to bring +G and -G together for the unpack
// (distributed_real_gamma.rs:651-682, 1316-1339). Representatives are in |G|
// order, so the 16-byte reads and writes of X and Y are scattered over the
// column: whole pairs go to one XCD, whose L2 then serves a column's lines to
// all its tiles.
//
// The kernels with one workgroup-wide pass per radix staged a tile of 32
// sticks in LDS, zeros included, with strides that repeat LDS banks at
// n0 = 72 and 144 and each column spread over all XCDs. Measured, FP64: 72^3,
// 80 pairs, into the sticks 121 -> 35 us and out of them 156 -> 33 us (94 MB
// of sticks and 31 or 62 MB of columns: 3.6 and 4.7 TB/s); 144^3, 563 pairs
// 6.3 -> 2.9 and 10.0 -> 3.3 ms; 135 x 72 x 72, 144 pairs 315 -> 128 and, adding
// to Y, 546 -> 114 us.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>

#include "common.hpp"
#include "op.hpp"
#include "stick.hpp"

namespace bd {
namespace {

constexpr double kSqrt2 = 1.41421356237309504880168872420969808;
constexpr double kInvSqrt2 = 0.70710678118654752440084436210484904;
// The LDS image leaves room for 4 waves a SIMD (FP64): registers for that many,
// so that a lane's loads are all issued before the first is waited for.
#define BD_WAVES(lo, hi) __attribute__((amdgpu_waves_per_eu(lo, hi)))
constexpr int kWaves = 4, kXcds = 8;

template <int A, int B>
struct Line {
  static constexpr int n = A * B, per = 64 / (A > B ? A : B), tile = kWaves * per;
  static constexpr int lx = A | 1;  // odd: neither side's stride repeats a bank
  static constexpr int row = (n > B * lx ? n : B * lx) | 1;
};

// Two doubles at 8-byte alignment (rows 2i - 1 and 2i of a column).
struct __attribute__((packed, aligned(8))) Rows2 {
  double re, im;
};

// LDS traffic between the lanes of one wavefront: its LDS instructions
// complete in order, so only the compiler has to be held back.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// (tile, pair) of this workgroup; false past the last.
template <typename F>
__device__ __forceinline__ bool place(const StickArgs<F>& a, int& tile, int& pair) {
  if (a.by_xcd) {
    const int q = int(blockIdx.x) / kXcds;
    tile = q % a.tiles;
    pair = q / a.tiles * kXcds + int(blockIdx.x) % kXcds;
  } else {
    tile = int(blockIdx.x) % a.tiles;
    pair = int(blockIdx.x) / a.tiles;
  }
  return pair < a.pairs;
}

template <typename F, int A, int B, bool K>
__global__ __launch_bounds__(64 * kWaves) BD_WAVES(2, 4) void k_stick_pair_inverse(StickArgs<F> a) {
  using S = Line<A, B>;
  __shared__ c2<F> image[S::tile * S::row];
  __shared__ c2<F> rt[S::n];
  int tile, t;
  if (!place(a, tile, t)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const bool hb = !K && 2 * t + 1 < a.m;
  const double* xa = a.x + int64_t(K ? t : 2 * t) * a.ldx;
  const double* xb = hb ? xa + a.ldx : xa;
  const int* ids = a.rep_at + ((int64_t(tile) * kWaves + wave) * A) * 64 + lane;
  int id[A];
#pragma unroll
  for (int r = 0; r < A; ++r) id[r] = ids[r * 64];
  for (int i = threadIdx.x; i < S::n; i += 64 * kWaves) rt[i] = {F(a.roots[i].x), F(a.roots[i].y)};
  const int l1 = lane / B, j1 = lane - l1 * B;
  const int l2 = lane / A, j2 = lane - l2 * A;
  c2<F> v[A];
  if (K) {
    double2 c[A];
#pragma unroll
    for (int r = 0; r < A; ++r)
      c[r] = *reinterpret_cast<const double2*>(xa + 2 * int64_t(id[r] > 0 ? id[r] - 1 : 0));
#pragma unroll
    for (int r = 0; r < A; ++r) {
      const double s = id[r] > 0 ? 1.0 : 0.0;
      v[r] = {F(s * c[r].x), F(s * c[r].y)};
    }
  } else {
    Rows2 pa[A], pb[A];
#pragma unroll
    for (int r = 0; r < A; ++r) {
      const int i = abs(id[r]) - 1;  // (none: -1)
      const int64_t at = i > 0 ? 2 * int64_t(i) - 1 : 0;
      pa[r] = *reinterpret_cast<const Rows2*>(xa + at);
      pb[r] = *reinterpret_cast<const Rows2*>(xb + at);
    }
    // +G: a + i b; -G: conj(a) + i conj(b). Selects by factors, so that the
    // loads above stay together.
#pragma unroll
    for (int r = 0; r < A; ++r) {
      const double one = id[r] == 1 ? 1.0 : 0.0;  // G = 0: row 0 alone, unscaled
      const double s = abs(id[r]) > 1 ? kInvSqrt2 : 0.0, sign = id[r] > 0 ? s : -s, both = hb ? 1.0 : 0.0;
      v[r] = {F((s + one) * pa[r].re - both * sign * pb[r].im), F(both * (s + one) * pb[r].re + sign * pa[r].im)};
    }
  }
  __syncthreads();  // the roots
  if (l1 < S::per) {
    dft<A, true>(v);
    c2<F>* w = image + (wave * S::per + l1) * S::row + j1 * S::lx;
#pragma unroll
    for (int r = 0; r < A; ++r) w[r] = v[r];
  }
  wave_sync();
  if (l2 < S::per) {
    const int slot = wave * S::per + l2;
    const c2<F>* w = image + slot * S::row + j2;
    c2<F> u[B];
#pragma unroll
    for (int r = 0; r < B; ++r) u[r] = w[r * S::lx];
#pragma unroll
    for (int r = 1; r < B; ++r) {
      const c2<F> z = rt[j2 * r];
      u[r] = cmul(u[r], c2<F>{z.x, -z.y});
    }
    dft<B, true>(u);
    c2<F>* out = a.sticks + (int64_t(t) * a.n0 + j2) * a.Spad + a.dst[tile * S::tile + slot];
#pragma unroll
    for (int r = 0; r < B; ++r) out[int64_t(A * r) * a.Spad] = u[r];
  }
}

template <typename F, int A, int B, StickOut OUT>
__global__ __launch_bounds__(64 * kWaves) BD_WAVES(2, 4) void k_stick_pair_forward(StickArgs<F> a) {
  using S = Line<A, B>;
  __shared__ c2<F> image[S::tile * S::row];
  __shared__ c2<F> rt[S::n];
  int tile, t;
  if (!place(a, tile, t)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int l1 = lane / B, j1 = lane - l1 * B;
  const int l2 = lane / A, j2 = lane - l2 * A;
  const int slot2 = wave * S::per + min(l2, S::per - 1);
  c2<F> u[B];
  {
    const c2<F>* in = a.sticks + (int64_t(t) * a.n0 + j2) * a.Spad + a.dst[tile * S::tile + slot2];
#pragma unroll
    for (int r = 0; r < B; ++r) u[r] = in[int64_t(A * r) * a.Spad];
  }
  for (int i = threadIdx.x; i < S::n; i += 64 * kWaves) rt[i] = {F(a.roots[i].x), F(a.roots[i].y)};
  const int e1 = a.tile_off[tile + 1];
  int e = a.tile_off[tile] + threadIdx.x;
  int4 en = e < e1 ? a.entries[e] : make_int4(0, 0, 0, 0);
  __syncthreads();  // the roots
  if (l2 < S::per) {
    dft<B, false>(u);
    c2<F>* w = image + slot2 * S::row + j2;
#pragma unroll
    for (int r = 0; r < B; ++r) w[r * S::lx] = u[r];
  }
  wave_sync();
  {
    c2<F>* line = image + (wave * S::per + min(l1, S::per - 1)) * S::row;
    c2<F> v[A];
    if (l1 < S::per) {
#pragma unroll
      for (int r = 0; r < A; ++r) v[r] = line[j1 * S::lx + r];
    }
    wave_sync();
    if (l1 < S::per) {
#pragma unroll
      for (int r = 1; r < A; ++r) v[r] = cmul(v[r], rt[j1 * r]);
      dft<A, false>(v);
#pragma unroll
      for (int r = 0; r < A; ++r) line[j1 + B * r] = v[r];
    }
  }
  constexpr bool ACC = OUT == StickOut::add;
  if (OUT == StickOut::k) {
    const double* x = a.x + int64_t(t) * a.ldx;
    double* y = a.y + int64_t(t) * a.ldy;
    __syncthreads();
    for (; e < e1; e += 64 * kWaves) {
      en = a.entries[e];
      const int64_t at = 2 * int64_t(en.x);
      const c2<F> h = image[en.y];
      const double2 v = *reinterpret_cast<const double2*>(x + at);
      const double k = a.kinetic[at];
      *reinterpret_cast<double2*>(y + at) =
          make_double2(double(h.x) * a.inv_n + k * v.x, double(h.y) * a.inv_n + k * v.y);
    }
    return;
  }
  const bool hb = 2 * t + 1 < a.m;
  const double* xa = a.x + int64_t(2 * t) * a.ldx;
  const double* xb = hb ? xa + a.ldx : xa;
  double* ya = a.y + int64_t(2 * t) * a.ldy;
  double* yb = hb ? ya + a.ldy : ya;
  const double* base_a = ACC ? ya : xa;  // what the local part is added to
  const double* base_b = ACC ? yb : xb;
  // Loads of an entry's rows run ahead of the barrier (the first) and of the
  // unpack (the later ones).
  double k = 0.0;
  Rows2 pa{0.0, 0.0}, pb{0.0, 0.0};
  auto fetch = [&]() {
    const int64_t at = en.x > 0 ? 2 * int64_t(en.x) - 1 : 0;
    pa = *reinterpret_cast<const Rows2*>(base_a + at);
    pb = *reinterpret_cast<const Rows2*>(base_b + at);
    if (!ACC) k = a.kinetic[at];
  };
  if (e < e1) fetch();
  __syncthreads();
  while (e < e1) {
    const int i = en.x;
    const c2<F> lp = image[en.y], lm = image[en.z];
    const double kk = ACC ? 1.0 : k;
    const Rows2 qa = pa, qb = pb;
    e += 64 * kWaves;
    if (e < e1) {
      en = a.entries[e];
      fetch();
    }
    const c2<double> hp = {double(lp.x) * a.inv_n, double(lp.y) * a.inv_n};
    const c2<double> hm = {double(lm.x) * a.inv_n, double(lm.y) * a.inv_n};
    if (i == 0) {
      ya[0] = hp.x + kk * qa.re;
      if (hb) yb[0] = hp.y + kk * qb.re;
    } else {
      // even = (hp + conj(hm))/2, odd = (hp - conj(hm))/2, rows x sqrt2.
      const double er = 0.5 * (hp.x + hm.x), ei = 0.5 * (hp.y - hm.y);
      const double orr = 0.5 * (hp.x - hm.x), oi = 0.5 * (hp.y + hm.y);
      const int64_t at = 2 * int64_t(i) - 1;
      *reinterpret_cast<Rows2*>(ya + at) = {er * kSqrt2 + kk * qa.re, ei * kSqrt2 + kk * qa.im};
      if (hb) *reinterpret_cast<Rows2*>(yb + at) = {oi * kSqrt2 + kk * qb.re, -orr * kSqrt2 + kk * qb.im};
    }
  }
}

// The 2,3,5-smooth lengths that are a product of two radices (A the larger).
#define BD_LINES(X)                                                                                          \
  X(5, 3) X(5, 4) X(6, 4) X(5, 5) X(9, 3) X(6, 5) X(8, 4) X(6, 6) X(8, 5) X(9, 5) X(8, 6) X(10, 5) X(9, 6)    \
  X(10, 6) X(8, 8) X(9, 8) X(15, 5) X(10, 8) X(9, 9) X(10, 9) X(12, 8) X(10, 10) X(12, 9) X(12, 10) X(16, 8) \
  X(15, 9) X(12, 12) X(15, 10) X(16, 10)

template <typename F>
using StickKernel = void (*)(StickArgs<F>);

template <typename F>
StickKernel<F> inverse_kernel(int n0, bool k) {
  switch (n0) {
#define BD_CASE(A, B) \
  case A * B:         \
    return k ? &k_stick_pair_inverse<F, A, B, true> : &k_stick_pair_inverse<F, A, B, false>;
    BD_LINES(BD_CASE)
#undef BD_CASE
  }
  return nullptr;
}

template <typename F, StickOut OUT>
StickKernel<F> forward_kernel(int n0) {
  switch (n0) {
#define BD_CASE(A, B) \
  case A * B:         \
    return &k_stick_pair_forward<F, A, B, OUT>;
    BD_LINES(BD_CASE)
#undef BD_CASE
  }
  return nullptr;
}

// Whole pairs to the XCDs where that leaves none of them more than a quarter
// short of work.
template <typename F>
unsigned grid(StickArgs<F>& a) {
  const int rounds = (a.pairs + kXcds - 1) / kXcds;
  a.by_xcd = 4 * rounds * kXcds <= 5 * a.pairs;
  return unsigned(a.tiles) * unsigned(a.by_xcd ? rounds * kXcds : a.pairs);
}
}  // namespace

StickShape stick_shape(int n0) {
  switch (n0) {
#define BD_CASE(A, B) \
  case A * B:         \
    return {true, A, B, Line<A, B>::per, Line<A, B>::tile, Line<A, B>::row};
    BD_LINES(BD_CASE)
#undef BD_CASE
  }
  return {};
}

template <typename F>
void stick_inverse(hipStream_t s, const StickShape& shape, StickArgs<F> a, bool k) {
  const StickKernel<F> f = inverse_kernel<F>(shape.a * shape.b, k);
  if (!f) fail(BD_ERR_APPLICATION, "no x-pass kernel");
  const unsigned blocks = grid(a);
  hipLaunchKernelGGL(f, dim3(blocks), dim3(64 * kWaves), 0, s, a);
}

template <typename F>
void stick_forward(hipStream_t s, const StickShape& shape, StickArgs<F> a, StickOut out) {
  const int n0 = shape.a * shape.b;
  const StickKernel<F> f = out == StickOut::h     ? forward_kernel<F, StickOut::h>(n0)
                           : out == StickOut::add ? forward_kernel<F, StickOut::add>(n0)
                                                  : forward_kernel<F, StickOut::k>(n0);
  if (!f) fail(BD_ERR_APPLICATION, "no x-pass kernel");
  const unsigned blocks = grid(a);
  hipLaunchKernelGGL(f, dim3(blocks), dim3(64 * kWaves), 0, s, a);
}

template void stick_inverse<double>(hipStream_t, const StickShape&, StickArgs<double>, bool);
template void stick_inverse<float>(hipStream_t, const StickShape&, StickArgs<float>, bool);
template void stick_forward<double>(hipStream_t, const StickShape&, StickArgs<double>, StickOut);
template void stick_forward<float>(hipStream_t, const StickShape&, StickArgs<float>, StickOut);

}  // namespace bd
