// FP64 tiled GEMM kernel on the matrix cores (v_mfma_f64_16x16x4f64).
//
// A workgroup of 4 waves makes a 64 RB x 16 NB tile; wave w owns the RB
// 16-row blocks from 16 RB w and all NB column blocks, so an A operand
// belongs to one wave and goes from global memory straight into its
// registers, and only B is shared, through LDS. Operands move as fragments of
// 16 indices x 8 k: lane l holds the pair k = 2 (l / 16), 2 (l / 16) + 1 of
// index l % 16, 16 bytes, which serves two MFMAs (the even k of the eight,
// then the odd ones; the sum over k may take any order). A B fragment is 1 KB
// of consecutive lanes in LDS: ds_write_b128 and ds_read_b128 without bank
// conflicts. The MFMA takes B as its row operand, so that a lane's results
// are consecutive rows of the column-major C across l % 16.
//
// Global loads run D slices (16 k each) ahead in registers, the B stages are
// double buffered, and one barrier a slice is left.
//
// CHAIN (Sums::chain): lane l's pair is k = l / 16 and l / 16 + 4, so that the two
// MFMAs take four ascending k each and every result is one ascending chain;
// the loads are then of 8 bytes.
//
// Bound: FP64 MFMA issue at the large shapes, the latency of a slice at the
// small ones. Measured against 64 x 64 tiles with both operands through LDS
// one slice ahead: A^T B of 2560 x 1126 x 191711 35.8 -> 19.3 ms (57 TFLOP/s),
// A B of 191711 x 1126 x 2560 27.5 -> 18.4 ms (60); 320 x 160 x 23847 91 -> 55
// us with its partial sums, 23847 x 160 x 320 89 -> 53 us. The split sums'
// error against compensated sums (2-norm): 7.4e-15 at K = 191711, where one
// chain over K has 2.0e-14.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace bd {
namespace gemm64 {

constexpr int TK = 16;  // k per slice: two fragments
typedef double f64x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
// Two doubles at 8-byte alignment (columns of odd leading dimension); global
// memory takes the 16-byte load at any dword.
struct __attribute__((packed, aligned(8))) Pair8 {
  double x, y;
};

template <int RB, int NB>
struct Tile {
  static constexpr int rows = 64 * RB, cols = 16 * NB;
  static constexpr int bfrags = 2 * NB;              // B fragments per slice
  static constexpr int bwave = (bfrags + 3) / 4;     // fragments a wave stages
  // Slices in flight: two where a slice is short against the memory latency.
  static constexpr int depth = RB * NB >= 8 ? 1 : 2;
  // Waves per SIMD the registers are kept for: the accumulators take 8 RB NB.
  static constexpr int waves = RB * NB >= 6 ? 2 : 3;
};

// One output tile: acc = sum over k in [kbeg, kend) of A[k, rows] B[k, cols].
// A: row i, index k at A[i + k lda] (TA = false) or A[k + i lda] (TA = true);
// B: k, column j at B[k + j ldb]. Rows past M and columns past N repeat the
// last one (their results are not stored); k past kend counts as zero.
template <int RB, int NB, bool TA, bool CHAIN = false>
__device__ __forceinline__ void tile_product(int64_t M, int64_t N, int64_t kbeg, int64_t kend, int64_t row0,
                                             int64_t col0, const double* __restrict__ A, int64_t lda,
                                             const double* __restrict__ B, int64_t ldb,
                                             f64x2 (*Bs)[Tile<RB, NB>::bfrags * 64], f64x4 (&acc)[RB][NB]) {
  using T = Tile<RB, NB>;
  constexpr int D = T::depth, BW = T::bwave;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lg = lane >> 4;
  constexpr int step = CHAIN ? 4 : 1;       // a lane's k: first and first + step
  const int first = CHAIN ? lg : 2 * lg;
#pragma unroll
  for (int r = 0; r < RB; ++r)
#pragma unroll
    for (int c = 0; c < NB; ++c) acc[r][c] = f64x4{0.0, 0.0, 0.0, 0.0};
  const double* pa[RB];
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int64_t i = min(row0 + (wave * RB + r) * 16 + li, M - 1);
    pa[r] = TA ? A + i * lda + first : A + i + first * lda;
  }
  // Fragment f = wave + 4 u of a slice: column block f / 2, k half f % 2.
  const double* pb[BW];
#pragma unroll
  for (int u = 0; u < BW; ++u) {
    const int f = min(wave + 4 * u, T::bfrags - 1);
    pb[u] = B + min(col0 + (f >> 1) * 16 + li, N - 1) * ldb + (f & 1) * 8 + first;
  }
  auto along_k = [](const double* p) {  // the pair where k is contiguous
    if (CHAIN) return f64x2{p[0], p[step]};
    const Pair8 v = *reinterpret_cast<const Pair8*>(p);
    return f64x2{v.x, v.y};
  };
  f64x2 ra[D][RB][2], rb[D][BW];
  auto fetch = [&](f64x2 (&a)[RB][2], f64x2 (&b)[BW], int64_t k0) {
#pragma unroll
    for (int u = 0; u < BW; ++u) b[u] = along_k(pb[u] + k0);
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        if (TA) {
          a[r][h] = along_k(pa[r] + k0 + 8 * h);
        } else {
          const double* p = pa[r] + (k0 + 8 * h) * lda;
          a[r][h] = f64x2{p[0], p[step * lda]};
        }
      }
  };
  auto stash = [&](const f64x2 (&b)[BW], int stage) {
#pragma unroll
    for (int u = 0; u < BW; ++u)
      if (wave + 4 * u < T::bfrags) Bs[stage][(wave + 4 * u) * 64 + lane] = b[u];
  };
  auto multiply = [&](const f64x2 (&a)[RB][2], int stage) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      f64x2 b[NB];
#pragma unroll
      for (int c = 0; c < NB; ++c) b[c] = Bs[stage][(2 * c + h) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 2; ++e)
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
          for (int r = 0; r < RB; ++r)
            acc[r][c] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[c][e], a[r][h][e], acc[r][c], 0, 0, 0);
    }
  };
  const int64_t full = (kend - kbeg) / TK;
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < full) fetch(ra[d], rb[d], kbeg + d * TK);
  // Stage s % 2 is rewritten at slice s + 2, after the barrier of slice
  // s + 1, which every wave reaches only when it is done with slice s.
  for (int64_t s = 0; s < full; s += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (s + d >= full) break;
      const int stage = int(s + d) & 1;
      stash(rb[d], stage);
      f64x2 a[RB][2];
#pragma unroll
      for (int r = 0; r < RB; ++r) {
        a[r][0] = ra[d][r][0];
        a[r][1] = ra[d][r][1];
      }
      if (s + d + D < full) fetch(ra[d], rb[d], kbeg + (s + d + D) * TK);
      __syncthreads();
      multiply(a, stage);
    }
  }
  const int64_t k0 = kbeg + full * TK;
  if (k0 < kend) {  // the ragged end, element by element
    f64x2 a[RB][2], b[BW];
#pragma unroll
    for (int u = 0; u < BW; ++u) {
      const int f = min(wave + 4 * u, T::bfrags - 1);
      const int64_t k = k0 + (f & 1) * 8 + first;
      b[u] = f64x2{k < kend ? pb[u][k0] : 0.0, k + step < kend ? pb[u][k0 + step] : 0.0};
    }
#pragma unroll
    for (int r = 0; r < RB; ++r)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        const int64_t k = k0 + 8 * h + first;
        const double* p = TA ? pa[r] + k0 + 8 * h : pa[r] + (k0 + 8 * h) * lda;
        a[r][h] = f64x2{k < kend ? p[0] : 0.0, k + step < kend ? p[TA ? step : step * lda] : 0.0};
      }
    const int stage = int(full) & 1;
    stash(b, stage);
    __syncthreads();
    multiply(a, stage);
  }
}

// Workgroups are dealt to the 8 XCDs round robin (id % 8); the logical index
// gives each XCD consecutive work: the tiles of one K chunk (TN) or the column
// tiles of a few row tiles (NN), which share that XCD's L2.
constexpr int kXcds = 8;
__device__ __forceinline__ int xcd_index(int total) {
  const int per_xcd = (total + kXcds - 1) / kXcds;
  return (int(blockIdx.x) % kXcds) * per_xcd + int(blockIdx.x) / kXcds;
}

// C = alpha A B + beta C (TA: A^T), the whole k range in one workgroup.
template <int RB, int NB, bool TA = false, bool CHAIN = false>
__global__ __launch_bounds__(256, (Tile<RB, NB>::waves)) void k_gemm_nn(int64_t M, int64_t N, int64_t K, int tiles_n,
                                                                      int total, double alpha,
                                                                      const double* __restrict__ A, int64_t lda,
                                                                      const double* __restrict__ B, int64_t ldb,
                                                                      double beta, double* __restrict__ C,
                                                                      int64_t ldc) {
  __shared__ f64x2 Bs[2][Tile<RB, NB>::bfrags * 64];
  const int logical = xcd_index(total);
  if (logical >= total) return;
  const int64_t row0 = int64_t(logical / tiles_n) * (64 * RB), col0 = int64_t(logical % tiles_n) * (16 * NB);
  f64x4 acc[RB][NB];
  tile_product<RB, NB, TA, CHAIN>(M, N, 0, K, row0, col0, A, lda, B, ldb, Bs, acc);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int64_t i = row0 + (wave * RB + r) * 16 + (lane & 15);
    if (i >= M) continue;
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t j = col0 + c * 16 + (lane >> 4) + 4 * v;
        if (j >= N) continue;
        double* p = C + i + j * ldc;
        *p = beta == 0.0 ? alpha * acc[r][c][v] : alpha * acc[r][c][v] + beta * *p;
      }
  }
}

// TN partial: part[s] (M x N) = sum over k in chunk s of A[k, i] B[k, j].
template <int RB, int NB, bool CHAIN = false>
__global__ __launch_bounds__(256, (Tile<RB, NB>::waves)) void k_gemm_tn(int64_t M, int64_t N, int64_t K, int64_t chunk,
                                                                      int tiles_m, int tiles, int total,
                                                                      const double* __restrict__ A, int64_t lda,
                                                                      const double* __restrict__ B, int64_t ldb,
                                                                      double* __restrict__ part) {
  __shared__ f64x2 Bs[2][Tile<RB, NB>::bfrags * 64];
  const int logical = xcd_index(total);
  if (logical >= total) return;
  const int tile = logical % tiles, kc = logical / tiles;
  const int64_t row0 = int64_t(tile % tiles_m) * (64 * RB), col0 = int64_t(tile / tiles_m) * (16 * NB);
  const int64_t kbeg = int64_t(kc) * chunk, kend = min(K, kbeg + chunk);
  f64x4 acc[RB][NB];
  tile_product<RB, NB, true, CHAIN>(M, N, kbeg, kend, row0, col0, A, lda, B, ldb, Bs, acc);
  double* out = part + int64_t(kc) * M * N;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int r = 0; r < RB; ++r) {
    const int64_t i = row0 + (wave * RB + r) * 16 + (lane & 15);
    if (i >= M) continue;
#pragma unroll
    for (int c = 0; c < NB; ++c)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int64_t j = col0 + c * 16 + (lane >> 4) + 4 * v;
        if (j < N) out[i + j * M] = acc[r][c][v];
      }
  }
}

// Products whose 64-row tiles would leave most CUs idle and whose k range is
// short (the m x m products of the subspace step): a 16 x 16 NB tile per
// workgroup, the k range split over its 4 waves, which read their fragments
// straight from global memory (L2) D steps of 8 k ahead and meet once at the
// end, where the four sums are added in wave order.
template <bool TA, int NB>
__global__ __launch_bounds__(256) void k_gemm_short(int64_t M, int64_t N, int64_t K, double alpha,
                                                    const double* __restrict__ A, int64_t lda,
                                                    const double* __restrict__ B, int64_t ldb, double beta,
                                                    double* __restrict__ C, int64_t ldc) {
  constexpr int D = 4;
  __shared__ double part[4][NB * 256];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lg = lane >> 4;
  const int64_t row0 = int64_t(blockIdx.x) * 16, col0 = int64_t(blockIdx.y) * (16 * NB);
  const int64_t span = ((K + 7) / 8 + 3) / 4 * 8;
  const int64_t kbeg = min(wave * span, K), kend = min(kbeg + span, K);
  const int64_t i = min(row0 + li, M - 1);
  const double* pa = TA ? A + i * lda + 2 * lg : A + i + 2 * lg * lda;
  const double* pb[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) pb[c] = B + min(col0 + c * 16 + li, N - 1) * ldb + 2 * lg;
  f64x4 acc[NB];
#pragma unroll
  for (int c = 0; c < NB; ++c) acc[c] = f64x4{0.0, 0.0, 0.0, 0.0};
  f64x2 ra[D], rb[D][NB];
  auto fetch = [&](f64x2& a, f64x2 (&b)[NB], int64_t k0) {
    if (TA) {
      const Pair8 v = *reinterpret_cast<const Pair8*>(pa + k0);
      a = f64x2{v.x, v.y};
    } else {
      a = f64x2{pa[k0 * lda], pa[(k0 + 1) * lda]};
    }
#pragma unroll
    for (int c = 0; c < NB; ++c) {
      const Pair8 v = *reinterpret_cast<const Pair8*>(pb[c] + k0);
      b[c] = f64x2{v.x, v.y};
    }
  };
  auto multiply = [&](const f64x2& a, const f64x2 (&b)[NB]) {
#pragma unroll
    for (int e = 0; e < 2; ++e)
#pragma unroll
      for (int c = 0; c < NB; ++c)
        acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[c][e], a[e], acc[c], 0, 0, 0);
  };
  const int64_t full = (kend - kbeg) / 8;
#pragma unroll
  for (int d = 0; d < D; ++d)
    if (d < full) fetch(ra[d], rb[d], kbeg + d * 8);
  for (int64_t s = 0; s < full; s += D) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (s + d >= full) break;
      multiply(ra[d], rb[d]);
      if (s + d + D < full) fetch(ra[d], rb[d], kbeg + (s + d + D) * 8);
    }
  }
  const int64_t k0 = kbeg + full * 8;
  if (k0 < kend) {  // the ragged end of the last wave's range
    const bool in0 = k0 + 2 * lg < kend, in1 = k0 + 2 * lg + 1 < kend;
    const double* p = TA ? pa + k0 : pa + k0 * lda;
    const f64x2 a = {in0 ? p[0] : 0.0, in1 ? p[TA ? 1 : lda] : 0.0};
    f64x2 b[NB];
#pragma unroll
    for (int c = 0; c < NB; ++c) b[c] = f64x2{in0 ? pb[c][k0] : 0.0, in1 ? pb[c][k0 + 1] : 0.0};
    multiply(a, b);
  }
#pragma unroll
  for (int c = 0; c < NB; ++c)
#pragma unroll
    for (int v = 0; v < 4; ++v) part[wave][c * 256 + (lg + 4 * v) * 16 + li] = acc[c][v];
  __syncthreads();
#pragma unroll
  for (int c = 0; c < NB; ++c) {
    const int e = c * 256 + threadIdx.x;
    const int64_t ci = row0 + (threadIdx.x & 15), cj = col0 + c * 16 + (threadIdx.x >> 4);
    if (ci >= M || cj >= N) continue;
    const double s = (part[0][e] + part[1][e]) + (part[2][e] + part[3][e]);
    double* p = C + ci + cj * ldc;
    *p = beta == 0.0 ? alpha * s : alpha * s + beta * *p;
  }
}

// C = alpha * (the partial sums in chunk order) + beta * C. Four threads an
// element, a quarter of the chunks each (eight loads in flight); CHAIN: one
// thread an element, all the chunks in order.
template <bool CHAIN = false>
__global__ __launch_bounds__(256) void k_gemm_reduce(int64_t M, int64_t N, int splits, double alpha,
                                                     const double* __restrict__ part, double beta,
                                                     double* __restrict__ C, int64_t ldc) {
  __shared__ double sum[4][64];
  const int lane = threadIdx.x & 63, q = threadIdx.x >> 6;
  const int64_t e = int64_t(blockIdx.x) * 64 + lane, total = M * N;
  const int per = CHAIN ? splits : (splits + 3) / 4, end = min(splits, (q + 1) * per);
  double s = 0.0;
  if (e < total) {
    int p = q * per;
    for (; p + 8 <= end; p += 8) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) v[u] = part[int64_t(p + u) * total + e];
#pragma unroll
      for (int u = 0; u < 8; ++u) s += v[u];
    }
    for (; p < end; ++p) s += part[int64_t(p) * total + e];
  }
  sum[q][lane] = s;
  __syncthreads();
  if (q != 0 || e >= total) return;
  if (!CHAIN) s = (sum[0][lane] + sum[1][lane]) + (sum[2][lane] + sum[3][lane]);
  double* c = C + e % M + (e / M) * ldc;
  *c = beta == 0.0 ? alpha * s : alpha * s + beta * *c;
}

}  // namespace gemm64
}  // namespace bd
