// The paired plane pass. A workgroup takes one (x, pair) plane: inverse y
// transforms of its Z occupied lines from the sticks into LDS, per y row the
// inverse z transform, * V(r) and the forward z transform, forward y
// transforms back to the sticks (distributed_fft.rs:956-1080).
//
// A line of n = ra * rb points is two radix passes. A wavefront owns whole
// lines: pass one does ra-point transforms (rb of them a line, one per lane),
// the values change lanes through LDS words that only this wavefront touches,
// pass two does rb-point transforms. The inverse ends and the forward
// transform begins with radix rb on the same elements j + ra r, so V is applied
// in registers between them: a row crosses LDS twice and reads and writes the
// plane once, where the pass-per-radix kernel (k_plane) crossed it eight times
// with a workgroup barrier at each. y lines change lanes in place, inside
// their own row of the plane.
//
// The rest of the design follows from the LDS: real and imaginary parts of a
// z row cross one after the other through the same words (half the space), so
// two workgroups of 6 wavefronts fit a CU at 72^2 planes. Where the plane is
// too large (144^2 in FP64) the even and the odd y rows are done in turn: a
// radix-2 step in y on the way in (a_k +- a_{k + n1/2}) and on the way out.
//
// Measured: 72^2 FP64, 80 pairs x 72 planes 248 us, bound by the LDS and FP64
// issue of 12 wavefronts a CU (673 KB of LDS traffic and 0.34 Mflop-lanes a
// plane: 50-60 us each); the pass-per-radix kernel took 809 us at its best
// shape and 1136 us at its default one. Density of 144 pairs x 135 planes
// 777 us (3829), kept fields 477 us (3417). 144^2 FP64, 563 pairs: 14.4 ms,
// where the planes through HBM took 103 ms.
#pragma once
#include <hip/hip_runtime.h>

#include "plane.hpp"

namespace bd {
namespace {

constexpr int kMaxWaves = 8;

// Wavefronts per SIMD the registers are held to: FP64 radices up to 10 need
// 162 at most, 12 and 16 up to 239; FP32 stays under 128.
template <typename F>
constexpr int waves_per_simd(int ya, int A) {
  return sizeof(F) == 4 ? 4 : (ya > 10 || A > 10) ? 2 : 3;
}


// LDS traffic between the lanes of one wavefront: its LDS instructions
// complete in order, so only the compiler has to be held back.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <typename F>
__device__ __forceinline__ c2<F> conj_if(c2<F> w, bool c) {
  return c ? c2<F>{w.x, -w.y} : w;
}

// Keeps what is computed from a lane's place inside the loop that uses it:
// hoisted out, a kernel's worth of addresses and predicates would spill.
__device__ __forceinline__ int here(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

// LDS row of a y line: its padded exchange layout fits, and an odd length
// keeps the z rows' column accesses off one another's banks.
__host__ __device__ constexpr int line_row(int ya, int yb) {
  return (ya * yb > yb * (ya | 1) ? ya * yb : yb * (ya | 1)) | 1;
}

// Rows of one wavefront and the LDS words they exchange through (z rows).
template <int A, int B>
struct RowShape {
  static constexpr int rows = 64 / (A > B ? A : B);
  static constexpr int lx = A | 1;  // odd: neither side's stride repeats a bank
  static constexpr int row = B * lx;
  static constexpr int words = rows * row;
};

// Move a row's values from writers (v, R1 of them, words wb + r ws) to readers
// (u, R2 of them, words rb + r rs), the two parts one after the other.
template <int R1, int R2, typename F>
__device__ __forceinline__ void exchange(F* xb, const c2<F>* v, bool aw, int wb, int ws, c2<F>* u, bool ar, int rb,
                                         int rs) {
  if (aw) {
#pragma unroll
    for (int r = 0; r < R1; ++r) xb[wb + r * ws] = v[r].x;
  }
  wave_sync();
  if (ar) {
#pragma unroll
    for (int r = 0; r < R2; ++r) u[r].x = xb[rb + r * rs];
  }
  wave_sync();
  if (aw) {
#pragma unroll
    for (int r = 0; r < R1; ++r) xb[wb + r * ws] = v[r].y;
  }
  wave_sync();
  if (ar) {
#pragma unroll
    for (int r = 0; r < R2; ++r) u[r].y = xb[rb + r * rs];
  }
  wave_sync();
}

// Inverse y transforms of every line: sticks -> P[line][0 .. ny).
template <typename F, int SPLIT, int ya, int yb>
__device__ __forceinline__ void y_inverse(const PairArgs<F>& a, const c2<F>* col, int parity, c2<F>* P,
                                          const c2<F>* rt) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  constexpr int ny = ya * yb, lx = ya | 1, n1 = ny * SPLIT, ldp = line_row(ya, yb);
  constexpr int per = 64 / (ya > yb ? ya : yb);
  for (int l0 = wave * per; l0 < a.Z; l0 += waves * per) {
    const int ln = here(lane);
    const int l1 = ln / yb, j1 = ln - l1 * yb;
    const int l2 = ln / ya, j2 = ln - l2 * ya;
    {
      const int line = l0 + l1;
      const bool on = l1 < per && line < a.Z;
      {
        constexpr int ra = ya;
        if (on) {
          const PlaneLine L = a.lines[line];
          const c2<F>* src = col + L.first;
          auto get = [&](int k) {
            int q = k - L.start;
            q += q < 0 ? n1 : 0;
            return q < L.count ? src[q] : c2<F>{F(0), F(0)};
          };
          c2<F> v[ra];
#pragma unroll
          for (int r = 0; r < ra; ++r) v[r] = get(j1 + yb * r);
          if (SPLIT == 2) {
#pragma unroll
            for (int r = 0; r < ra; ++r) {
              const int k = j1 + yb * r;
              const c2<F> h = get(k + ny);
              v[r] = parity ? cmul(csub(v[r], h), conj_if(rt[k], true)) : cadd(v[r], h);
            }
          }
          dft<ra, true>(v);
          c2<F>* dst = P + line * ldp + j1 * lx;
#pragma unroll
          for (int r = 0; r < ra; ++r) dst[r] = v[r];
        }
      }
    }
    wave_sync();
    {
      const int line = l0 + l2;
      const bool on = l2 < per && line < a.Z;
      {
        constexpr int rb = yb;
        c2<F> u[rb];
        c2<F>* row = P + line * ldp + j2;
        if (on) {
#pragma unroll
          for (int r = 0; r < rb; ++r) u[r] = row[r * lx];
        }
        wave_sync();
        if (on) {
          const int ts = j2 * SPLIT;
#pragma unroll
          for (int r = 1; r < rb; ++r) u[r] = cmul(u[r], conj_if(rt[ts * r], true));
          dft<rb, true>(u);
#pragma unroll
          for (int r = 0; r < rb; ++r) row[r * ya] = u[r];
        }
      }
    }
    wave_sync();
  }
}

// Forward y transforms of every line: P -> sticks.
template <typename F, int SPLIT, int ya, int yb>
__device__ __forceinline__ void y_forward(const PairArgs<F>& a, c2<F>* col, int parity, c2<F>* P, const c2<F>* rt) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  constexpr int ny = ya * yb, lx = ya | 1, n1 = ny * SPLIT, ldp = line_row(ya, yb);
  constexpr int per = 64 / (ya > yb ? ya : yb);
  for (int l0 = wave * per; l0 < a.Z; l0 += waves * per) {
    const int ln = here(lane);
    const int l1 = ln / yb, j1 = ln - l1 * yb;
    const int l2 = ln / ya, j2 = ln - l2 * ya;
    {
      const int line = l0 + l2;
      const bool on = l2 < per && line < a.Z;
      {
        constexpr int rb = yb;
        c2<F> u[rb];
        c2<F>* row = P + line * ldp + j2;
        if (on) {
#pragma unroll
          for (int r = 0; r < rb; ++r) u[r] = row[r * ya];
        }
        wave_sync();
        if (on) {
          dft<rb, false>(u);
#pragma unroll
          for (int r = 0; r < rb; ++r) row[r * lx] = u[r];
        }
      }
    }
    wave_sync();
    {
      const int line = l0 + l1;
      const bool on = l1 < per && line < a.Z;
      {
        constexpr int ra = ya;
        if (on) {
          const c2<F>* row = P + line * ldp + j1 * lx;
          const int ts = j1 * SPLIT;
          c2<F> v[ra];
#pragma unroll
          for (int r = 0; r < ra; ++r) v[r] = row[r];
#pragma unroll
          for (int r = 1; r < ra; ++r) v[r] = cmul(v[r], rt[ts * r]);
          dft<ra, false>(v);
          const PlaneLine L = a.lines[line];
          c2<F>* dst = col + L.first;
#pragma unroll
          for (int r = 0; r < ra; ++r) {
            const int k = j1 + yb * r;
            int q = k - L.start;
            q += q < 0 ? n1 : 0;
            if (SPLIT == 1) {
              if (q < L.count) dst[q] = v[r];
            } else {
              // Even rows give E for k and k + ny, odd rows +- w^k O.
              int q2 = k + ny - L.start;
              q2 += q2 < 0 ? n1 : 0;
              if (!parity) {
                if (q < L.count) dst[q] = v[r];
                if (q2 < L.count) dst[q2] = v[r];
              } else {
                const c2<F> o = cmul(v[r], rt[k]);
                if (q < L.count) dst[q] = cadd(dst[q], o);
                if (q2 < L.count) dst[q2] = csub(dst[q2], o);
              }
            }
          }
        }
      }
    }
    wave_sync();
  }
}

// z rows of the plane. MODE 0: inverse, * V, forward. MODE 1: inverse and the
// band density. MODE 2: kept field * dV, forward.
template <int MODE, typename F, int SPLIT, int ya, int yb, int A, int B>
__device__ __forceinline__ void z_rows(const PairArgs<F>& a, int xi, int t, int parity, double wa, double wb,
                                       bool first, double* rho, c2<F>* P, F* xb, const c2<F>* rt) {
  using S = RowShape<A, B>;
  constexpr int n2 = A * B;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
  constexpr int ny = ya * yb, n1 = ny * SPLIT, ldp = line_row(ya, yb);
  for (int y0 = wave * S::rows; y0 < ny; y0 += waves * S::rows) {
    const int ln = here(lane);
    const int r1 = ln / B, j1 = ln - r1 * B;  // A-point transforms: elements j1 + B r
    const int r2 = ln / A, j2 = ln - r2 * A;  // B-point transforms: elements j2 + A r
    const int ra = y0 + r1, rb = y0 + r2;
    const bool on1 = r1 < S::rows && ra < ny, on2 = r2 < S::rows && rb < ny;
    // Row rb of the whole plane, its first element of this lane.
    const int64_t at = ((int64_t(xi) * n1) + int64_t(rb) * SPLIT + parity) * n2 + j2;
    c2<F> u[B];
    F pot[B];
    if (MODE != 1 && on2) {
#pragma unroll
      for (int r = 0; r < B; ++r) pot[r] = a.potential[at + A * r];
    }
    if (MODE != 2) {
      c2<F> v[A];
      if (on1) {
#pragma unroll
        for (int r = 0; r < A; ++r) {
          int q = j1 + B * r - a.zs;
          q += q < 0 ? n2 : 0;
          v[r] = q < a.Z ? P[q * ldp + ra] : c2<F>{F(0), F(0)};
        }
        dft<A, true>(v);
      }
      exchange<A, B>(xb, v, on1, r1 * S::row + j1 * S::lx, 1, u, on2, r2 * S::row + j2, S::lx);
      if (on2) {
#pragma unroll
        for (int r = 1; r < B; ++r) u[r] = cmul(u[r], conj_if(rt[j2 * r], true));
        dft<B, true>(u);
      }
    } else if (on2) {
      const c2<F>* kp = a.kept_in + int64_t(t) * a.n0 * n1 * n2 + at;
#pragma unroll
      for (int r = 0; r < B; ++r) u[r] = kp[A * r];
    }
    if (MODE == 1) {
      if (on2) {
        double* out = rho + at;
        c2<F>* kp = a.kept_out ? a.kept_out + int64_t(t) * a.n0 * n1 * n2 + at : nullptr;
#pragma unroll
        for (int r = 0; r < B; ++r) {
          const double re = double(u[r].x), im = double(u[r].y);
          const double d = wa * re * re + wb * im * im;
          out[A * r] = first ? d : out[A * r] + d;
          if (kp) kp[A * r] = u[r];
        }
      }
    } else {
      c2<F> v[A];
      if (on2) {
#pragma unroll
        for (int r = 0; r < B; ++r) u[r] = cscale(u[r], pot[r]);
        dft<B, false>(u);
      }
      exchange<B, A>(xb, u, on2, r2 * S::row + j2, S::lx, v, on1, r1 * S::row + j1 * S::lx, 1);
      if (on1) {
#pragma unroll
        for (int r = 1; r < A; ++r) v[r] = cmul(v[r], rt[j1 * r]);
        dft<A, false>(v);
#pragma unroll
        for (int r = 0; r < A; ++r) {
          int q = j1 + B * r - a.zs;
          q += q < 0 ? n2 : 0;
          if (q < a.Z) P[q * ldp + ra] = v[r];
        }
      }
    }
  }
}

// MODE 0 and 2: grid (pairs, n0). MODE 1: grid (n0, groups); group g sums the
// pairs g, g + groups, ... in order into its partial grid.
template <int MODE, typename F, int SPLIT, int ya, int yb, int A, int B>
__global__ __launch_bounds__(64 * kMaxWaves, waves_per_simd<F>(ya, A)) void k_plane_pair(PairArgs<F> a) {
  extern __shared__ __attribute__((aligned(16))) char smem[];
  c2<F>* P = reinterpret_cast<c2<F>*>(smem);
  constexpr int n1 = ya * yb * SPLIT, n2 = A * B;
  c2<F>* rty = P + a.Z * line_row(ya, yb);
  c2<F>* rtz = rty + n1;
  F* xb = reinterpret_cast<F*>(rtz + n2) + (threadIdx.x >> 6) * RowShape<A, B>::words;
  for (int i = threadIdx.x; i < n1; i += blockDim.x) rty[i] = {F(a.roots[a.n0 + i].x), F(a.roots[a.n0 + i].y)};
  for (int i = threadIdx.x; i < n2; i += blockDim.x)
    rtz[i] = {F(a.roots[a.n0 + n1 + i].x), F(a.roots[a.n0 + n1 + i].y)};
  __syncthreads();
  const int xi = MODE == 1 ? blockIdx.x : blockIdx.y;
  const int tbeg = MODE == 1 ? blockIdx.y : blockIdx.x;
  const int tend = MODE == 1 ? a.pairs : tbeg + 1;
  const int step = MODE == 1 ? gridDim.y : 1;
  double* rho = MODE == 1 ? a.rho + int64_t(blockIdx.y) * a.n0 * n1 * n2 : nullptr;
  for (int t = tbeg; t < tend; t += step) {
    const int64_t col = (int64_t(t) * a.n0 + xi) * a.Spad;
    double wa = 0.0, wb = 0.0;
    if (MODE == 1) {
      wa = a.weights[2 * t] * a.inv_volume;
      wb = a.weights[2 * t + 1] * a.inv_volume;
    }
    for (int p = 0; p < SPLIT; ++p) {
      if (MODE != 2) {
        y_inverse<F, SPLIT, ya, yb>(a, a.in + col, p, P, rty);
        __syncthreads();
      }
      z_rows<MODE, F, SPLIT, ya, yb, A, B>(a, xi, t, p, wa, wb, t == tbeg, rho, P, xb, rtz);
      __syncthreads();
      if (MODE != 1) {
        y_forward<F, SPLIT, ya, yb>(a, a.out + col, p, P, rty);
        if (p + 1 < SPLIT) __syncthreads();
      }
    }
  }
}

// The planes the kernels are built for, as X(split, ya, yb, A, B) with
// n1 = split ya yb and n2 = A B: the larger radix outside (A, ya), the radix
// whose z transform runs twice around V inside (B). Equal axes of 15 to 48, 54,
// 60, 64, 72, 80, 90, 96, 108, 120, 128 and 144 points; 128^2 and 144^2 also by
// row parity (FP64 planes beyond one workgroup's LDS); and unequal axes of
// supercells one, two and three cells long at 30, 32 and 36 points a cell. A
// kernel is compiled for each plane, mode and type: other planes (50, 75, 81,
// 100, 135 points, other unequal axes) run the pass-per-radix kernels.
#define BD_PLANES(X)                                                                                  \
  X(1, 5, 3, 5, 3) X(1, 5, 4, 5, 4) X(1, 6, 4, 6, 4) X(1, 5, 5, 5, 5) X(1, 9, 3, 9, 3)                \
  X(1, 6, 5, 6, 5) X(1, 8, 4, 8, 4) X(1, 6, 6, 6, 6) X(1, 8, 5, 8, 5) X(1, 9, 5, 9, 5)                \
  X(1, 8, 6, 8, 6) X(1, 9, 6, 9, 6) X(1, 10, 6, 10, 6) X(1, 8, 8, 8, 8) X(1, 9, 8, 9, 8)              \
  X(1, 10, 8, 10, 8) X(1, 10, 9, 10, 9) X(1, 12, 8, 12, 8) X(1, 12, 9, 12, 9) X(1, 12, 10, 12, 10)    \
  X(1, 16, 8, 16, 8) X(1, 12, 12, 12, 12) X(2, 8, 8, 16, 8) X(2, 9, 8, 12, 12)                        \
  X(1, 6, 5, 10, 6) X(1, 10, 6, 6, 5) X(1, 10, 6, 10, 9) X(1, 10, 9, 10, 6) X(1, 6, 5, 10, 9)         \
  X(1, 10, 9, 6, 5) X(1, 8, 4, 8, 8) X(1, 8, 8, 8, 4) X(1, 8, 8, 12, 8) X(1, 12, 8, 8, 8)             \
  X(1, 8, 4, 12, 8) X(1, 12, 8, 8, 4) X(1, 6, 6, 9, 8) X(1, 9, 8, 6, 6) X(1, 9, 8, 12, 9)             \
  X(1, 12, 9, 9, 8) X(1, 6, 6, 12, 9) X(1, 12, 9, 6, 6)

template <typename F>
using PairKernel = void (*)(PairArgs<F>);

constexpr int plane_key(int split, int n1, int n2) { return (split * 1024 + n1) * 1024 + n2; }

}  // namespace

template <typename F, int MODE>
const void* pair_kernel(int split, int n1, int n2) {
  PairKernel<F> k = nullptr;
  switch (plane_key(split, n1, n2)) {
#define BD_CASE(SPLIT, YA, YB, A, B)                  \
  case plane_key(SPLIT, SPLIT * YA * YB, A * B):      \
    k = &k_plane_pair<MODE, F, SPLIT, YA, YB, A, B>; \
    break;
    BD_PLANES(BD_CASE)
#undef BD_CASE
  }
  return reinterpret_cast<const void*>(k);
}

template const void* pair_kernel<BD_PLANE_TYPE, BD_PLANE_MODE>(int, int, int);

#ifdef BD_PLANE_LAYOUTS
bool plane_layout(int split, int n1, int n2, PlaneLayout& out) {
  switch (plane_key(split, n1, n2)) {
#define BD_CASE(SPLIT, YA, YB, A, B)                                                                      \
  case plane_key(SPLIT, SPLIT * YA * YB, A * B):                                                          \
    out = {line_row(YA, YB), RowShape<A, B>::words, RowShape<A, B>::rows, waves_per_simd<double>(YA, A), \
           waves_per_simd<float>(YA, A)};                                                                 \
    return true;
    BD_PLANES(BD_CASE)
#undef BD_CASE
  }
  return false;
}
#endif

}  // namespace bd
