// k-point H·X of one column in one workgroup with every line as two
// in-register radix passes of one wavefront (equal axes of n = A B points,
// the lengths of plane_kernels.hpp and stick.hip whose columns fit the LDS).
// The column's sticks stay in LDS; a wavefront transforms sticks and then
// whole y-z planes by itself, in its own plane buffer, so the workgroup meets
// four times a column where one workgroup-wide pass per radix
// (k_hpsi_fused) met some twenty times every few planes. The arithmetic of a
// line, V and the kinetic term are those of the paired stick/plane path: the
// local part has its bits. One launch covers every column of every k point of
// a batch, nonlocal term included, as k_hpsi_fused does.
//
// Measured, Al 4-atom cell (25^3, 936 to 955 coefficients, 32 projector
// columns, 108 k points): 160 us a launch of the Davidson's columns (its mean
// over a map), 1028 us with the radix-pass kernel. Bound by LDS and FP64
// issue of the 8 wavefronts that a CU's LDS holds (46 KB of sticks a column).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <string>

#include "common.hpp"
#include "op.hpp"

namespace bd {
namespace {

constexpr size_t kLdsMax = 160 * 1024;

template <int A, int B>
struct Cube {
  static constexpr int n = A * B, per = 64 / (A > B ? A : B);
  static constexpr int lx = A | 1;                          // odd: neither side's stride repeats a bank
  static constexpr int row = (n > B * lx ? n : B * lx) | 1;  // a stick or a y line
  static constexpr int words = per * B * lx;                // z rows: one part at a time
};

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Keeps what is computed from a lane's place inside the loop that uses it.
__device__ __forceinline__ int here(int v) {
  asm volatile("" : "+v"(v));
  return v;
}

template <typename F>
__device__ __forceinline__ c2<F> conj_of(c2<F> w) {
  return {w.x, -w.y};
}

// The two parts of a z row change lanes one after the other.
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

__device__ __forceinline__ int find_item(const KWork* __restrict__ works, int count, int item) {
  int lo = 0, hi = count - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (works[mid].first <= item) lo = mid;
    else hi = mid - 1;
  }
  return lo;
}

// One y-z plane of the column by one wavefront: the sticks' values at x = xi
// (L[stick * row + xi]) -> inverse y and z, * V, forward z and y -> back.
template <typename F, int A, int B>
__device__ __forceinline__ void plane(const KWork& w, c2<F>* L, int xi, const F* __restrict__ pot, c2<F>* P, F* xb,
                                      const c2<F>* rt) {
  using S = Cube<A, B>;
  const int lane = threadIdx.x & 63;
  for (int l0 = 0; l0 < w.Z; l0 += S::per) {
    const int ln = here(lane);
    const int l1 = ln / B, j1 = ln - l1 * B;
    const int l2 = ln / A, j2 = ln - l2 * A;
    {
      const int line = l0 + l1;
      if (l1 < S::per && line < w.Z) {
        const PlaneLine pl = w.lines[line];
        c2<F> v[A];
#pragma unroll
        for (int r = 0; r < A; ++r) {
          int q = j1 + B * r - pl.start;
          q += q < 0 ? S::n : 0;
          v[r] = q < pl.count ? L[(pl.first + q) * S::row + xi] : c2<F>{F(0), F(0)};
        }
        dft<A, true>(v);
        c2<F>* dst = P + line * S::row + j1 * S::lx;
#pragma unroll
        for (int r = 0; r < A; ++r) dst[r] = v[r];
      }
    }
    wave_sync();
    {
      const int line = l0 + l2;
      const bool on = l2 < S::per && line < w.Z;
      c2<F> u[B];
      c2<F>* row = P + line * S::row + j2;
      if (on) {
#pragma unroll
        for (int r = 0; r < B; ++r) u[r] = row[r * S::lx];
      }
      wave_sync();
      if (on) {
#pragma unroll
        for (int r = 1; r < B; ++r) u[r] = cmul(u[r], conj_of(rt[j2 * r]));
        dft<B, true>(u);
#pragma unroll
        for (int r = 0; r < B; ++r) row[r * A] = u[r];
      }
    }
    wave_sync();
  }
  for (int y0 = 0; y0 < S::n; y0 += S::per) {
    const int ln = here(lane);
    const int r1 = ln / B, j1 = ln - r1 * B;
    const int r2 = ln / A, j2 = ln - r2 * A;
    const int ra = y0 + r1, rb = y0 + r2;
    const bool on1 = r1 < S::per && ra < S::n, on2 = r2 < S::per && rb < S::n;
    c2<F> u[B], v[A];
    F vr[B];
    if (on2) {
#pragma unroll
      for (int r = 0; r < B; ++r) vr[r] = pot[(xi * S::n + rb) * S::n + j2 + A * r];
    }
    if (on1) {
#pragma unroll
      for (int r = 0; r < A; ++r) {
        int q = j1 + B * r - w.zs;
        q += q < 0 ? S::n : 0;
        v[r] = q < w.Z ? P[q * S::row + ra] : c2<F>{F(0), F(0)};
      }
      dft<A, true>(v);
    }
    const int at1 = (r1 * B + j1) * S::lx, at2 = r2 * B * S::lx + j2;
    exchange<A, B>(xb, v, on1, at1, 1, u, on2, at2, S::lx);
    if (on2) {
#pragma unroll
      for (int r = 1; r < B; ++r) u[r] = cmul(u[r], conj_of(rt[j2 * r]));
      dft<B, true>(u);
#pragma unroll
      for (int r = 0; r < B; ++r) u[r] = cscale(u[r], vr[r]);
      dft<B, false>(u);
    }
    exchange<B, A>(xb, u, on2, at2, S::lx, v, on1, at1, 1);
    if (on1) {
#pragma unroll
      for (int r = 1; r < A; ++r) v[r] = cmul(v[r], rt[j1 * r]);
      dft<A, false>(v);
#pragma unroll
      for (int r = 0; r < A; ++r) {
        int q = j1 + B * r - w.zs;
        q += q < 0 ? S::n : 0;
        if (q < w.Z) P[q * S::row + ra] = v[r];
      }
    }
  }
  wave_sync();
  for (int l0 = 0; l0 < w.Z; l0 += S::per) {
    const int ln = here(lane);
    const int l1 = ln / B, j1 = ln - l1 * B;
    const int l2 = ln / A, j2 = ln - l2 * A;
    {
      const int line = l0 + l2;
      const bool on = l2 < S::per && line < w.Z;
      c2<F> u[B];
      c2<F>* row = P + line * S::row + j2;
      if (on) {
#pragma unroll
        for (int r = 0; r < B; ++r) u[r] = row[r * A];
      }
      wave_sync();
      if (on) {
        dft<B, false>(u);
#pragma unroll
        for (int r = 0; r < B; ++r) row[r * S::lx] = u[r];
      }
    }
    wave_sync();
    {
      const int line = l0 + l1;
      if (l1 < S::per && line < w.Z) {
        const c2<F>* row = P + line * S::row + j1 * S::lx;
        c2<F> v[A];
#pragma unroll
        for (int r = 0; r < A; ++r) v[r] = row[r];
#pragma unroll
        for (int r = 1; r < A; ++r) v[r] = cmul(v[r], rt[j1 * r]);
        dft<A, false>(v);
        const PlaneLine pl = w.lines[line];
#pragma unroll
        for (int r = 0; r < A; ++r) {
          int q = j1 + B * r - pl.start;
          q += q < 0 ? S::n : 0;
          if (q < pl.count) L[(pl.first + q) * S::row + xi] = v[r];
        }
      }
    }
    wave_sync();
  }
}

// Persistent: workgroup b takes items b, b + grid, ...; every workgroup leaves
// after its last item.
template <typename F, int A, int B>
__global__ __launch_bounds__(512, 2) void k_hpsi_pair(const KWork* __restrict__ works, KWork one, int count, int total,
                                                      const c2<double>* __restrict__ roots, int qmax, double inv_n) {
  using S = Cube<A, B>;
  extern __shared__ __attribute__((aligned(16))) char smem[];
  const int nt = blockDim.x, waves = nt >> 6;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  c2<F>* rt = reinterpret_cast<c2<F>*>(smem);
  double* nlq = reinterpret_cast<double*>(rt + S::n + (S::n & 1));
  double* nlw = nlq + qmax;
  c2<F>* L = reinterpret_cast<c2<F>*>(nlw + qmax);  // S sticks of `row`
  for (int i = tid; i < S::n; i += nt) rt[i] = {F(roots[i].x), F(roots[i].y)};
  for (int item = blockIdx.x; item < total; item += gridDim.x) {
    const KWork w = works ? works[find_item(works, count, item)] : one;
    const int j = item - w.first, nk = w.nk, np2 = w.np2;
    const int64_t nr = 2 * int64_t(nk);
    c2<F>* P = L + w.S * S::row + wave * w.Z * S::row;
    F* xb = reinterpret_cast<F*>(L + (w.S + waves * w.Z) * S::row) + wave * S::words;
    const double* xc = w.x + int64_t(j) * w.ldx;
    double* yc = w.y + int64_t(j) * w.ldy;
    const F* pot = reinterpret_cast<const F*>(w.potential);
    __syncthreads();  // the roots; the previous item's last use of LDS
    // X -> sticks, inverse x.
    for (int g = wave; g * S::per < w.S; g += waves) {
      const int ln = here(lane);
      const int l1 = ln / B, j1 = ln - l1 * B;
      const int l2 = ln / A, j2 = ln - l2 * A;
      const int s1 = g * S::per + l1, s2 = g * S::per + l2;
      int id[A];
#pragma unroll
      for (int r = 0; r < A; ++r) id[r] = w.rep_at[(int64_t(g) * A + r) * 64 + ln];
      double2 c[A];
#pragma unroll
      for (int r = 0; r < A; ++r)
        c[r] = *reinterpret_cast<const double2*>(xc + 2 * int64_t(id[r] > 0 ? id[r] - 1 : 0));
      if (l1 < S::per && s1 < w.S) {
        c2<F> v[A];
#pragma unroll
        for (int r = 0; r < A; ++r) {
          const double s = id[r] > 0 ? 1.0 : 0.0;
          v[r] = {F(s * c[r].x), F(s * c[r].y)};
        }
        dft<A, true>(v);
        c2<F>* row = L + s1 * S::row + j1 * S::lx;
#pragma unroll
        for (int r = 0; r < A; ++r) row[r] = v[r];
      }
      wave_sync();
      c2<F>* row = L + s2 * S::row + j2;
      const bool on = l2 < S::per && s2 < w.S;
      c2<F> u[B];
      if (on) {
#pragma unroll
        for (int r = 0; r < B; ++r) u[r] = row[r * S::lx];
      }
      wave_sync();
      if (on) {
#pragma unroll
        for (int r = 1; r < B; ++r) u[r] = cmul(u[r], conj_of(rt[j2 * r]));
        dft<B, true>(u);
#pragma unroll
        for (int r = 0; r < B; ++r) row[A * r] = u[r];
      }
    }
    // Nonlocal q = P2^T x (FP64): eight projector columns a wavefront and
    // pass, two rows a lane, their loads together.
    for (int c0 = 8 * wave; c0 < np2; c0 += 8 * waves) {
      double acc[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc[u] = 0.0;
      for (int64_t r = 2 * lane; r < nr; r += 128) {
        const double2 xv = *reinterpret_cast<const double2*>(xc + r);
        double2 p[8];
#pragma unroll
        for (int u = 0; u < 8; ++u)
          p[u] = *reinterpret_cast<const double2*>(w.proj2 + int64_t(min(c0 + u, np2 - 1)) * nr + r);
#pragma unroll
        for (int u = 0; u < 8; ++u) acc[u] += p[u].x * xv.x + p[u].y * xv.y;
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        double s = acc[u];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
        if (lane == 0 && c0 + u < np2) nlq[c0 + u] = s;
      }
    }
    __syncthreads();
    for (int c = tid; c < np2; c += nt) {
      const int start = (c / w.nc) * w.nc, a = c - start;
      double v = 0.0;
      for (int b = 0; b < w.nc; ++b) v += w.blockd[a * w.nc + b] * nlq[start + b];
      nlw[c] = v;
    }
    for (int xi = wave; xi < S::n; xi += waves) plane<F, A, B>(w, L, xi, pot, P, xb, rt);
    __syncthreads();
    // Forward x.
    for (int g = wave; g * S::per < w.S; g += waves) {
      const int ln = here(lane);
      const int l1 = ln / B, j1 = ln - l1 * B;
      const int l2 = ln / A, j2 = ln - l2 * A;
      const int s1 = g * S::per + l1, s2 = g * S::per + l2;
      const bool on1 = l1 < S::per && s1 < w.S, on2 = l2 < S::per && s2 < w.S;
      c2<F>* row2 = L + s2 * S::row + j2;
      c2<F> u[B], v[A];
      if (on2) {
#pragma unroll
        for (int r = 0; r < B; ++r) u[r] = row2[A * r];
      }
      wave_sync();
      if (on2) {
        dft<B, false>(u);
#pragma unroll
        for (int r = 0; r < B; ++r) row2[r * S::lx] = u[r];
      }
      wave_sync();
      c2<F>* row1 = L + s1 * S::row;
      if (on1) {
#pragma unroll
        for (int r = 0; r < A; ++r) v[r] = row1[j1 * S::lx + r];
      }
      wave_sync();
      if (on1) {
#pragma unroll
        for (int r = 1; r < A; ++r) v[r] = cmul(v[r], rt[j1 * r]);
        dft<A, false>(v);
#pragma unroll
        for (int r = 0; r < A; ++r) row1[j1 + B * r] = v[r];
      }
      wave_sync();
    }
    __syncthreads();
    // 1/N, + |k+G|^2/2 x + P2 w.
    for (int g = tid; g < nk; g += nt) {
      const int64_t r = 2 * int64_t(g);
      const c2<F> h = L[w.fpos_row[g]];
      const double2 v = *reinterpret_cast<const double2*>(xc + r);
      const double k = w.kinetic[r];
      double y0 = double(h.x) * inv_n + k * v.x, y1 = double(h.y) * inv_n + k * v.y;
      if (np2 > 0) {
        double a0 = 0.0, a1 = 0.0;
        const double* p = w.proj2 + r;
        int c = 0;
        for (; c + 8 <= np2; c += 8) {
          double2 q[8];
#pragma unroll
          for (int u = 0; u < 8; ++u) q[u] = *reinterpret_cast<const double2*>(p + int64_t(c + u) * nr);
#pragma unroll
          for (int u = 0; u < 8; ++u) {
            a0 += q[u].x * nlw[c + u];
            a1 += q[u].y * nlw[c + u];
          }
        }
        for (; c < np2; ++c) {
          const double2 q = *reinterpret_cast<const double2*>(p + int64_t(c) * nr);
          a0 += q.x * nlw[c];
          a1 += q.y * nlw[c];
        }
        y0 += a0;
        y1 += a1;
      }
      *reinterpret_cast<double2*>(yc + r) = make_double2(y0, y1);
    }
  }
}

// Cubes up to 45 points (beyond, no column fits the LDS), radices as in the
// stick and plane kernels.
#define BD_CUBES(X) X(5, 3) X(5, 4) X(6, 4) X(5, 5) X(9, 3) X(6, 5) X(8, 4) X(6, 6) X(8, 5) X(9, 5)

template <typename F>
using CubeKernel = void (*)(const KWork*, KWork, int, int, const c2<double>*, int, double);

struct CubeSize {
  int row = 0, words = 0;
};

bool cube_size(int n, CubeSize& c) {
  switch (n) {
#define BD_CASE(A, B) \
  case A * B:         \
    c = {Cube<A, B>::row, Cube<A, B>::words}; \
    return true;
    BD_CUBES(BD_CASE)
#undef BD_CASE
  }
  return false;
}

template <typename F>
CubeKernel<F> cube_kernel(int n) {
  switch (n) {
#define BD_CASE(A, B) \
  case A * B:         \
    return &k_hpsi_pair<F, A, B>;
    BD_CUBES(BD_CASE)
#undef BD_CASE
  }
  return nullptr;
}

size_t cube_lds(const CubeSize& c, int n, int S, int Z, int np2, int waves, size_t elem) {
  return size_t(n + (n & 1) + (S + waves * Z) * c.row) * elem + size_t(waves) * c.words * (elem / 2) +
         size_t(2 * (np2 + (np2 & 1))) * sizeof(double);
}

// Wavefronts of a workgroup: as many a CU as fit, four where that is level.
int cube_waves(const CubeSize& c, int n, int S, int Z, int np2, size_t elem) {
  int best = 0, most = 0;
  for (int waves : {4, 8, 2, 1}) {
    const size_t lds = cube_lds(c, n, S, Z, np2, waves, elem);
    if (lds > kLdsMax) continue;
    const int on_cu = std::min(8, int(kLdsMax / lds) * waves);  // (8: the registers)
    if (on_cu > most) {
      most = on_cu;
      best = waves;
    }
  }
  return best;
}

template <typename F>
void launch(const GammaOp& op, const KPairShape& f, const KWork* works, const KWork& one, int count, int total,
            hipStream_t s) {
  const CubeKernel<F> k = cube_kernel<F>(op.plan.n0);
  if (!k || f.lds > kLdsMax || f.waves < 1) fail(BD_ERR_APPLICATION, "paired k kernel shape");
  static std::mutex mu;
  static bool raised[64] = {};
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!raised[op.plan.n0]) {
      BD_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                 int(kLdsMax)));
      raised[op.plan.n0] = true;
    }
  }
  // Workgroups past the resident ones take items in turn.
  const int per_cu = std::max(1, std::min(8 / f.waves, int(kLdsMax / f.lds)));
  const int grid = std::max(1, std::min(total, 256 * per_cu));
  const int qmax = int(op.nproj + (op.nproj & 1));
  hipLaunchKernelGGL(k, dim3(grid), dim3(64 * f.waves), f.lds, s, works, one, count, total, op.d_roots.p, qmax,
                     1.0 / double(op.N));
  BD_HIP(hipGetLastError());
}
}  // namespace

KPairShape kpair_shape(const StickPlan& p, int nproj, size_t elem) {
  KPairShape f;
  CubeSize c;
  if (p.n0 != p.n1 || p.n0 != p.n2 || p.lines.empty() || !cube_size(p.n0, c)) return f;
  f.waves = cube_waves(c, p.n0, p.S, p.Z, nproj, elem);
  f.on = f.waves > 0;
  if (f.on) f.lds = cube_lds(c, p.n0, p.S, p.Z, nproj, f.waves, elem);
  return f;
}

// One launch over several ops: the fewest wavefronts any of them takes, LDS
// for the largest; off where an op has no paired kernel.
KPairShape kpair_common(const GammaOp* const* ops, int count) {
  KPairShape f = ops[0]->kpair;
  for (int i = 1; i < count && f.on; ++i) {
    f.on = ops[i]->kpair.on;
    f.waves = std::min(f.waves, ops[i]->kpair.waves);
  }
  if (!f.on) return KPairShape{};
  CubeSize c;
  cube_size(ops[0]->plan.n0, c);
  f.lds = 0;
  for (int i = 0; i < count; ++i)
    f.lds = std::max(f.lds, cube_lds(c, ops[i]->plan.n0, ops[i]->plan.S, ops[i]->plan.Z, int(ops[i]->nproj), f.waves,
                                     ops[i]->elem_bytes()));
  return f;
}

void kpair_launch(const GammaOp& op, const KPairShape& f, const KWork* works, const KWork& one, int count, int total,
                  hipStream_t s) {
  if (total <= 0) return;
  if (op.fft32()) launch<float>(op, f, works, one, count, total, s);
  else launch<double>(op, f, works, one, count, total, s);
}

}  // namespace bd
