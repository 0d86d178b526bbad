// Bordered inverse Cholesky of the Davidson overlap and the small matrix
// helpers of the subspace step, on the GPU in FP64.
//
// extend_inverse_cholesky_dev follows crates/dft-solvers/src/lean_davidson.rs:
// 167-331: with T11 = L11^{-1} known for the leading `from` columns of S,
//   W = T11 S12,  G = S22 - W^T W = L22 L22^T,  T22 = L22^{-1},
//   T21 = -T22 W^T T11,
// rejecting when a squared pivot over its overlap diagonal falls below
// eps/1e-12 (or is NaN), or when a new row of T fails the growth test
// eps * (sum_j |T_ij| sqrt(S_jj))^2 <= sqrt(eps).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <string>

#include "common.hpp"
#include "eigen.hpp"
#include "gemm.hpp"

namespace bd {

namespace {
constexpr int kCT = 1024;
constexpr int kInvRows = 2;  // k_chol_inv_lds: rows a lane (k <= 128)
constexpr double kPivotRatioMin = DBL_EPSILON / 1e-12;  // lean_davidson.rs:62-64

// Lane l's value of v (l uniform across the wave).
__device__ __forceinline__ double read_lane(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}

__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

// G (k x k, ld k) <- S[from:to, from:to].
__global__ void k_copy_block(int k, const double* __restrict__ S, int64_t lds, double* __restrict__ G) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i < k) G[i + int64_t(j) * k] = S[i + int64_t(j) * lds];
}

// Cholesky of the k x k block G (k <= 64 * kInvRows) with the pivot-ratio
// test, then T22 = L^{-1} into T (ld ldt), zero above the diagonal. A flag
// already set by an earlier block of the same border leaves the block
// untouched; min_ratio keeps the minimum over the blocks.
//
// G = M D M^T with M unit lower: column l sits in the registers of wave
// l mod 16 (lane i owns row i, and i + 64 past 64 rows), and a step passes one column
// through LDS: one barrier, one division. The pivots are tested together at
// the end (a failed one only spoils later columns, which nobody then reads).
// M^{-1} by forward substitution, a wave's columns side by side so that their
// chains (a lane read and the update) overlap; L^{-1} = D^{-1/2} M^{-1}.
// CHAIN (Sums::chain, GammaOp::keeps_rounding): the rounding of G = L L^T, L's
// columns those of the elimination over sqrt(d_j), the substitution on L.
// Bound by the chain of steps. k = 80: 51 us, k = 20: 7 (CHAIN 60 and 8); 98 and
// 16, with CHAIN's bits, with the block as a packed triangle in LDS, two
// divisions a step and one column at a time in the substitution.
template <int NC, bool CHAIN>
__global__ __launch_bounds__(kCT) void k_chol_inv_lds(int k, const double* __restrict__ G,
                                                      const double* __restrict__ sdiag, int64_t sstride,
                                                      double* __restrict__ T22, int64_t ldt, int* __restrict__ flag,
                                                      double* __restrict__ min_ratio) {
  extern __shared__ double sh[];
  if (flag[0]) return;  // an earlier block of this border failed: uniform exit
  // NC columns a wave; rows a lane.
  constexpr int nw = kCT / 64, R = NC * nw <= 64 ? 1 : 2;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ldm = k + 1;
  double* M = sh;                        // k columns of ldm
  double* pass = M + int64_t(k) * ldm;   // two slots of k: the column of a step
  double* dv = pass + 2 * k;             // k: the pivots (CHAIN: then 1 / sqrt of them)
  double a[NC][R];
  int row[R];  // this lane's rows, the last one's for those past it
#pragma unroll
  for (int t = 0; t < R; ++t) row[t] = min(lane + 64 * t, k - 1);
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int t = 0; t < R; ++t) {
      const int l = wave + nw * c, i = lane + 64 * t;
      a[c][t] = l < k && i < k && i >= l ? G[i + int64_t(l) * k] : 0.0;
    }
#pragma unroll
  for (int jc = 0; jc < NC; ++jc)
    for (int jw = 0; jw < nw; ++jw) {
      const int j = jc * nw + jw;
      if (j >= k) break;
      double* col = pass + (j & 1) * k;
      if (wave == jw) {
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const int i = lane + 64 * t;
          if (i < k) col[i] = a[jc][t];
          if (i == j) dv[j] = a[jc][t];
        }
      }
      __syncthreads();
      // (Columns up to j take the update too; nothing reads them again.)
      const double dj = col[j];
      double mine[R], alj[NC];
#pragma unroll
      for (int t = 0; t < R; ++t) mine[t] = col[row[t]];
#pragma unroll
      for (int c = jc; c < NC; ++c) alj[c] = col[min(wave + nw * c, k - 1)];
      const double inv_d = 1.0 / dj;
      if (CHAIN) {
#pragma unroll
        for (int c = jc; c < NC; ++c) alj[c] *= inv_d;
      } else {
#pragma unroll
        for (int t = 0; t < R; ++t) mine[t] *= inv_d;
      }
#pragma unroll
      for (int c = jc; c < NC; ++c)
#pragma unroll
        for (int t = 0; t < R; ++t) a[c][t] = fma(-mine[t], alj[c], a[c][t]);
      if (wave == jw) {
#pragma unroll
        for (int t = 0; t < R; ++t) {
          const int i = lane + 64 * t;
          if (i < k) M[i + int64_t(j) * ldm] = i > j ? mine[t] : 0.0;
        }
      }
    }
  __syncthreads();
  // The pivots' ratios, up to the first that fails.
  double mr = INFINITY;
  bool failed = false, nan = false;
  for (int j0 = 0; j0 < k && !failed; j0 += 64) {
    const int j = j0 + lane;
    const double ratio = j < k ? dv[j] / sdiag[int64_t(j) * sstride] : INFINITY;
    const unsigned long long bad = __ballot(isnan(ratio) || ratio < kPivotRatioMin);
    const int first = bad ? __ffsll(static_cast<long long>(bad)) - 1 : 63;
    double r = lane <= first ? ratio : INFINITY;
    nan = bad && isnan(__shfl(ratio, first, 64));
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) r = fmin(r, __shfl_xor(r, off, 64));
    mr = fmin(mr, r);
    failed = bad != 0;
  }
  if (tid == 0) {
    min_ratio[0] = nan ? 0.0 : fmin(min_ratio[0], mr);
    if (failed) flag[0] = 1;
  }
  if (failed) return;  // every wave found the same: uniform exit
  if (CHAIN) {  // M = L below the diagonal
    for (int l = wave; l < k; l += nw) {
      const double sd = sqrt(dv[l]);
      for (int i = l + 1 + lane; i < k; i += 64) M[i + int64_t(l) * ldm] /= sd;
    }
    __syncthreads();
    for (int l = tid; l < k; l += kCT) dv[l] = 1.0 / sqrt(dv[l]);
    __syncthreads();
  }
  double x[NC][R], ml[R], rl = CHAIN ? dv[0] : 1.0;  // (M is zero up to the diagonal)
#pragma unroll
  for (int t = 0; t < R; ++t) {
    ml[t] = M[row[t]];
#pragma unroll
    for (int c = 0; c < NC; ++c) x[c][t] = lane + 64 * t == wave + nw * c ? 1.0 : 0.0;
  }
#pragma unroll
  for (int tl = 0; tl < R; ++tl) {
    const int end = min(k, 64 * (tl + 1));
    for (int l = 64 * tl; l < end; ++l) {
      double next[R];
#pragma unroll
      for (int t = 0; t < R; ++t) next[t] = M[row[t] + int64_t(min(l + 1, k - 1)) * ldm];
      const double next_rl = CHAIN ? dv[min(l + 1, k - 1)] : 1.0;
#pragma unroll
      for (int c = 0; c < NC; ++c) {
        const double xl = CHAIN ? read_lane(x[c][tl], l - 64 * tl) * rl : read_lane(x[c][tl], l - 64 * tl);
#pragma unroll
        for (int t = 0; t < R; ++t) x[c][t] = fma(-ml[t], xl, x[c][t]);
      }
#pragma unroll
      for (int t = 0; t < R; ++t) ml[t] = next[t];
      rl = next_rl;
    }
  }
#pragma unroll
  for (int t = 0; t < R; ++t) {
    const int i = lane + 64 * t;
    if (i >= k) continue;
    const double rs = CHAIN ? dv[i] : 1.0 / sqrt(dv[i]);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      const int l = wave + nw * c;
      if (l < k) T22[i + int64_t(l) * ldt] = i >= l ? x[c][t] * rs : 0.0;
    }
  }
}

typedef void (*CholInv)(int, const double*, const double*, int64_t, double*, int64_t, int*, double*);
template <bool CHAIN>
CholInv chol_inv_kernel(int k) {
  switch ((k * 64 + kCT - 1) / kCT) {  // columns a wave
    case 1: return &k_chol_inv_lds<1, CHAIN>;
    case 2: return &k_chol_inv_lds<2, CHAIN>;
    case 3: return &k_chol_inv_lds<3, CHAIN>;
    case 4: return &k_chol_inv_lds<4, CHAIN>;
    case 5: return &k_chol_inv_lds<5, CHAIN>;
    case 6: return &k_chol_inv_lds<6, CHAIN>;
    case 7: return &k_chol_inv_lds<7, CHAIN>;
    case 8: return &k_chol_inv_lds<8, CHAIN>;
  }
  return nullptr;
}

// One wave per new row i of T: finiteness and the growth guard.
__global__ __launch_bounds__(256) void k_growth_guard(const double* __restrict__ S, const double* __restrict__ T,
                                                      int cap, int from, int to, int guard, int* __restrict__ flag) {
  const int lane = threadIdx.x & 63;
  const int i = from + blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= to) return;
  double g = 0.0;
  int bad = 0;
  for (int j = lane; j <= i; j += 64) {
    const double v = T[i + int64_t(j) * cap];
    bad |= !isfinite(v);
    g += fabs(v) * sqrt(S[j + int64_t(j) * cap]);
  }
  g = wave_sum(g);
  if (lane == 0 && guard && (bad || !isfinite(g) || DBL_EPSILON * g * g > sqrt(DBL_EPSILON))) flag[0] = 1;
  if (bad) flag[0] = 1;
}

__global__ void k_mirror(double* __restrict__ M, int cap, int from, int to) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = from + blockIdx.y;
  if (j < to && i < j) M[j + int64_t(i) * cap] = M[i + int64_t(j) * cap];
}

__global__ void k_transpose(int m, int n, const double* __restrict__ A, int64_t lda, double* __restrict__ B,
                            int64_t ldb) {
  __shared__ double tile[32][33];
  const int bx = blockIdx.x * 32, by = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8 threads
  for (int r = ty; r < 32; r += 8) {
    const int i = bx + tx, j = by + r;
    if (i < m && j < n) tile[r][tx] = A[i + int64_t(j) * lda];
  }
  __syncthreads();
  for (int r = ty; r < 32; r += 8) {
    const int j = by + tx, i = bx + r;
    if (i < m && j < n) B[j + int64_t(i) * ldb] = tile[tx][r];
  }
}

__global__ void k_symmetrize(int m, double* __restrict__ A, int64_t lda) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i < j && j < m) {
    const double v = 0.5 * (A[i + int64_t(j) * lda] + A[j + int64_t(i) * lda]);
    A[i + int64_t(j) * lda] = v;
    A[j + int64_t(i) * lda] = v;
  }
}

__global__ void k_identity(int m, int n, double* __restrict__ A, int64_t lda) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x, j = blockIdx.y;
  if (i < m && j < n) A[i + int64_t(j) * lda] = i == j ? 1.0 : 0.0;
}

__global__ void k_zero_flag(int* flag, double* min_ratio) {
  flag[0] = 0;
  min_ratio[0] = INFINITY;
}
}  // namespace

// Partial sums of the products above (M, N, K <= cap): up to K = 1023 at most
// max(1, K / 256) copies of an M x N block; beyond, up to eight copies or 2^21
// values (max_splits of gemm.hip), of which cap / 256 >= 4 copies of cap x cap
// hold either. gemm_tn_work is monotone, so its value at cap covers them all.
int64_t factor_gwork(int cap) {
  const int64_t size = int64_t(cap < 256 ? 1 : cap / 256) * cap * cap;
  if (size < gemm_tn_work(cap, cap, cap)) fail(BD_ERR_APPLICATION, "factor workspace below its products' partial sums");
  return size;
}

namespace {
// Widest border block k_chol_inv_lds holds: its rows live in the kInvRows
// registers of a lane, and k(k + 1) + 3k doubles fit the 160 KB of LDS.
constexpr int kFactorBlock = 64 * kInvRows;
// Widest block a border is split into: the elimination costs ~k^3 / 3 in
// barriered column steps, so narrower blocks plus the extension GEMMs cost less.
constexpr int kFactorSplit = 96;

// T[from:to, 0:to] for one block of at most kFactorBlock new columns:
// W = T11 S12, G = S22 - W^T W, T22 = chol(G)^{-1}, T21 = -T22 W^T T11.
void extend_block(hipStream_t s, const double* S, double* T, int cap, int from, int to, const FactorWork& fw) {
  const int k = to - from;
  if (from > 0) fw.gemm.nn64(s, from, k, from, 1.0, T, cap, S + int64_t(from) * cap, cap, 0.0, fw.W, from);
  hipLaunchKernelGGL(k_copy_block, dim3((k + 255) / 256, k), dim3(256), 0, s, k,
                     S + from + int64_t(from) * cap, int64_t(cap), fw.G);
  if (from > 0) fw.gemm.tn64(s, k, k, from, -1.0, fw.W, from, fw.W, from, 1.0, fw.G, k, fw.gwork);
  double* T22 = T + from + int64_t(from) * cap;
  const size_t lds = (size_t(k) * (k + 1) + 3 * size_t(k)) * 8;
  if (k > kFactorBlock || lds > 160 * 1024) fail(BD_ERR_INVALID_PARAMETER, "inverse Cholesky block too large");
  const CholInv chol = fw.gemm.sums == Sums::chain ? chol_inv_kernel<true>(k) : chol_inv_kernel<false>(k);
  if (lds > 64 * 1024) allow_full_lds(reinterpret_cast<const void*>(chol), "k_chol_inv_lds");
  hipLaunchKernelGGL(chol, dim3(1), dim3(kCT), lds, s, k, fw.G, S + from + int64_t(from) * cap,
                     int64_t(cap) + 1, T22, int64_t(cap), fw.flag, fw.min_ratio);
  if (from > 0) {
    fw.gemm.tn64(s, k, from, from, 1.0, fw.W, from, T, cap, 0.0, fw.U, k, fw.gwork);  // U = W^T T11
    fw.gemm.nn64(s, k, from, k, -1.0, T22, cap, fw.U, k, 0.0, T + from, cap);          // T21 = -T22 U
  }
  hipLaunchKernelGGL(k_growth_guard, dim3((k + 3) / 4), dim3(256), 0, s, S, T, cap, from, to, fw.growth_guard,
                     fw.flag);
}
}  // namespace

// A border wider than one block is factored as successive extensions in
// near-equal blocks: the inverse Cholesky factor of S[0:b, 0:b] extended by
// the next columns of S is that of S[0:b', 0:b'] (the pivot of each column is
// the same Schur complement, so the pivot-ratio test is unchanged).
void extend_inverse_cholesky_dev(hipStream_t s, const double* S, double* T, int cap, int from, int to,
                                 const FactorWork& fw) {
  const int k = to - from;
  hipLaunchKernelGGL(k_zero_flag, dim3(1), dim3(1), 0, s, fw.flag, fw.min_ratio);
  if (k <= 0) return;
  const int blocks = (k + kFactorSplit - 1) / kFactorSplit;
  const int width = (k + blocks - 1) / blocks;
  for (int a = from; a < to; a += width) extend_block(s, S, T, cap, a, std::min(to, a + width), fw);
}

void mirror_border(hipStream_t s, double* M, int cap, int from, int to) {
  if (to <= from) return;
  hipLaunchKernelGGL(k_mirror, dim3((to + 255) / 256, to - from), dim3(256), 0, s, M, cap, from, to);
}

void transpose(hipStream_t s, int m, int n, const double* A, int64_t lda, double* B, int64_t ldb) {
  if (m <= 0 || n <= 0) return;
  hipLaunchKernelGGL(k_transpose, dim3((m + 31) / 32, (n + 31) / 32), dim3(256), 0, s, m, n, A, lda, B, ldb);
}

void symmetrize(hipStream_t s, int m, double* A, int64_t lda) {
  if (m <= 1) return;
  hipLaunchKernelGGL(k_symmetrize, dim3((m + 255) / 256, m), dim3(256), 0, s, m, A, lda);
}

void set_identity(hipStream_t s, int m, int n, double* A, int64_t lda) {
  if (m <= 0 || n <= 0) return;
  hipLaunchKernelGGL(k_identity, dim3((m + 255) / 256, n), dim3(256), 0, s, m, n, A, lda);
}

}  // namespace bd

namespace bd {
namespace {
// Factor scratch of one call at capacity cap: W, G, U (cap x cap each), the
// split-K partials, then min_ratio and the flag.
constexpr int64_t factor_scratch_doubles(int cap) {
  return 3 * int64_t(cap) * cap + int64_t(cap < 256 ? 1 : cap / 256) * cap * cap + 2;
}

FactorWork factor_layout(double* base, int cap) {
  const int64_t c2 = int64_t(cap) * cap;
  FactorWork fw;
  fw.W = base;
  fw.G = fw.W + c2;
  fw.U = fw.G + c2;
  fw.gwork = fw.U + c2;
  fw.min_ratio = fw.gwork + factor_gwork(cap);
  fw.flag = reinterpret_cast<int*>(fw.min_ratio + 1);
  return fw;
}

// One border extension on the null stream with its scratch at `base`; the
// verdict and the smallest pivot ratio are read back (synchronous).
void factor_on_null_stream(const double* S, double* T, int cap, int from, int to, double* base,
                           int32_t* accepted, double* min_ratio) {
  const FactorWork fw = factor_layout(base, cap);
  extend_inverse_cholesky_dev(nullptr, S, T, cap, from, to, fw);
  int flag = 0;
  if (hipMemcpy(&flag, fw.flag, sizeof(int), hipMemcpyDeviceToHost) != hipSuccess ||
      hipMemcpy(min_ratio, fw.min_ratio, sizeof(double), hipMemcpyDeviceToHost) != hipSuccess)
    fail(BD_ERR_DEVICE, "inverse Cholesky launch failed");
  *accepted = flag == 0 ? 1 : 0;
}

// Allocation-free variant: the scratch of every call on a GPU is this
// file-scope device array (each GPU holds its own copy until the process
// ends). Its host-side name is not a device address: kernels get the address
// from hipGetSymbolAddress, taken once per device with that device current.
// Calls that overlap on one GPU share the array and race.
constexpr int kStaticFactorCap = 640;
constexpr int64_t kStaticFactorDoubles = factor_scratch_doubles(kStaticFactorCap);
static __device__ __align__(256) double scratch[kStaticFactorDoubles];

constexpr int kMaxDevices = 64;
std::mutex scratch_mu;
double* scratch_dev[kMaxDevices] = {};

double* static_factor_scratch() {
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) fail(BD_ERR_DEVICE, "no current HIP device");
  if (dev < 0 || dev >= kMaxDevices) fail(BD_ERR_DEVICE, "device ordinal beyond the scratch table");
  std::lock_guard<std::mutex> lock(scratch_mu);
  if (!scratch_dev[dev]) {
    void* ptr = nullptr;
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr)
      fail(BD_ERR_DEVICE, std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e));
    scratch_dev[dev] = static_cast<double*>(ptr);
  }
  return scratch_dev[dev];
}
}  // namespace
}  // namespace bd

extern "C" bd_status bd_inverse_cholesky_dev(const double* S, double* T, int32_t cap, int32_t from, int32_t to,
                                             int32_t* accepted, double* min_ratio) {
  struct Scratch {
    double* p = nullptr;
    ~Scratch() {
      if (p) (void)hipFree(p);
    }
  } buf;
  BD_GUARD({
    if (!S || !T || !accepted || !min_ratio || cap <= 0 || from < 0 || to < from || to > cap)
      bd::fail(BD_ERR_INVALID_PARAMETER, "inverse Cholesky arguments");
    const int64_t total = bd::factor_scratch_doubles(cap);
    if (hipMalloc(&buf.p, size_t(total) * sizeof(double)) != hipSuccess) bd::fail(BD_ERR_DEVICE, "scratch");
    bd::factor_on_null_stream(S, T, cap, from, to, buf.p, accepted, min_ratio);
  });
}

extern "C" bd_status bd_inverse_cholesky_static_dev(const double* S, double* T, int32_t cap, int32_t from,
                                                    int32_t to, int32_t* accepted, double* min_ratio) {
  BD_GUARD({
    if (!S || !T || !accepted || !min_ratio || cap <= 0 || from < 0 || to < from || to > cap)
      bd::fail(BD_ERR_INVALID_PARAMETER, "inverse Cholesky arguments");
    if (cap > bd::kStaticFactorCap)
      bd::fail(BD_ERR_INVALID_PARAMETER, "bd_inverse_cholesky_static_dev: cap " + std::to_string(cap) +
                                             " exceeds the static scratch limit of " +
                                             std::to_string(bd::kStaticFactorCap));
    double* base = bd::static_factor_scratch();
    bd::factor_on_null_stream(S, T, cap, from, to, base, accepted, min_ratio);
  });
}
