// FP64 GEMMs: the choice of a tile and a split for each shape (the kernels are
// in gemm_f64.hpp), and the C entry points.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <string>
#include <type_traits>

#include "common.hpp"
#include "gemm.hpp"
#include "gemm_f64.hpp"

namespace bd {

namespace {
using gemm64::f64x4;

// Lane-layout probe: D (16x16, row-major) = A (16x4, row-major) B (4x16,
// row-major) by one v_mfma_f64_16x16x4f64 with the operand layout above.
__global__ void k_mfma_f64_probe(const double* __restrict__ A, const double* __restrict__ B, double* __restrict__ D) {
  const int lane = threadIdx.x;
  const double a = A[(lane & 15) * 4 + (lane >> 4)];
  const double b = B[(lane >> 4) * 16 + (lane & 15)];
  f64x4 d = {0.0, 0.0, 0.0, 0.0};
  d = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, d, 0, 0, 0);
  for (int v = 0; v < 4; ++v) D[((lane >> 4) + 4 * v) * 16 + (lane & 15)] = d[v];
}

// Tiles built: 64 rb x 16 nb.
struct TileShape {
  int rb, nb;
};
constexpr TileShape kTiles[] = {{1, 1}, {1, 2}, {1, 3}, {1, 5}, {1, 6}, {2, 2}, {2, 3}, {2, 4}, {2, 6}, {2, 8}};

// Cycles a CU needs for `wgs` tiles of `slices` 16-k slices, dealt evenly: 4 rb
// nb MFMAs of 64 cycles a slice on each SIMD (320 with the clock's drop under
// FP64 load), what a slice costs besides, and the latency that a slice leaves
// open when the CU's other workgroups are few. Within 15% of the measured
// times from 320 x 160 x 23847 to 191711 x 1126 x 2560.
double tile_cycles(const TileShape& t, int64_t wgs, int64_t slices) {
  const int64_t rounds = (wgs + 255) / 256;
  return double(slices) * (double(rounds) * (320.0 * t.rb * t.nb + 200.0) + 1000.0);
}

int64_t tiles_of(const TileShape& t, int64_t M, int64_t N) {
  return ((M + 64 * t.rb - 1) / (64 * t.rb)) * ((N + 16 * t.nb - 1) / (16 * t.nb));
}

// Products with a short k range and a small C run on k_gemm_short: below this
// the tiles fill too few CUs (NN 320 x 320 x 320: 5.6 us against 9.6 with the
// best tile, 320 x 160 x 320: 4.1 against 9.5); 640 x 640 x 640 is level.
bool short_product(int64_t M, int64_t N, int64_t K) {
  return K <= 1024 && ((M + 15) / 16) * ((N + 15) / 16) <= 800;
}

template <bool TA>
void launch_short(hipStream_t s, int64_t M, int64_t N, int64_t K, double alpha, const double* A, int64_t lda,
                  const double* B, int64_t ldb, double beta, double* C, int64_t ldc) {
  // 32-wide tiles where they still give most CUs a workgroup.
  const int64_t rows = (M + 15) / 16;
  if (rows * ((N + 31) / 32) >= 192)
    hipLaunchKernelGGL((gemm64::k_gemm_short<TA, 2>), dim3(unsigned(rows), unsigned((N + 31) / 32)), dim3(256), 0, s,
                       M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
  else
    hipLaunchKernelGGL((gemm64::k_gemm_short<TA, 1>), dim3(unsigned(rows), unsigned((N + 15) / 16)), dim3(256), 0, s,
                       M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
}

template <typename F>
void with_tile(const TileShape& t, const F& f) {
  switch (t.rb * 16 + t.nb) {
    case 17: return f(std::integral_constant<int, 1>(), std::integral_constant<int, 1>());
    case 18: return f(std::integral_constant<int, 1>(), std::integral_constant<int, 2>());
    case 19: return f(std::integral_constant<int, 1>(), std::integral_constant<int, 3>());
    case 21: return f(std::integral_constant<int, 1>(), std::integral_constant<int, 5>());
    case 22: return f(std::integral_constant<int, 1>(), std::integral_constant<int, 6>());
    case 34: return f(std::integral_constant<int, 2>(), std::integral_constant<int, 2>());
    case 35: return f(std::integral_constant<int, 2>(), std::integral_constant<int, 3>());
    case 36: return f(std::integral_constant<int, 2>(), std::integral_constant<int, 4>());
    case 38: return f(std::integral_constant<int, 2>(), std::integral_constant<int, 6>());
    case 40: return f(std::integral_constant<int, 2>(), std::integral_constant<int, 8>());
  }
  fail(BD_ERR_APPLICATION, "gemm tile");
}

unsigned xcd_grid(int64_t total) {
  if (total > (int64_t(1) << 30)) fail(BD_ERR_INVALID_PARAMETER, "gemm shape too large");
  return unsigned((total + gemm64::kXcds - 1) / gemm64::kXcds * gemm64::kXcds);
}

// Most K chunks a split product may take: 64 k at least in each and partial
// sums of at most 16 MB, or eight copies of C where that is more (four slices
// of k in a short range: the factor's products count on K / 256 there).
int64_t max_splits(int64_t M, int64_t N, int64_t K) {
  const int64_t few = std::max<int64_t>(1, std::min<int64_t>(K / 256, 8));
  if (K < 1024) return few;
  return std::min<int64_t>(K / 64, std::max(few, (int64_t(1) << 21) / (M * N)));
}

struct TnPlan {
  TileShape tile;
  int64_t chunk;
  int splits;
};

// The tile and split with the fewest cycles: the tiles' own, and the partial
// sums written and read (in part in cache) at about 2,300 bytes a cycle.
TnPlan tn_plan(int64_t M, int64_t N, int64_t K) {
  TnPlan best{kTiles[0], K, 1};
  double least = -1.0;
  const int64_t most = max_splits(M, N, K);
  for (const TileShape& t : kTiles) {
    const int64_t tiles = tiles_of(t, M, N);
    for (int64_t fill = 1; fill <= 8; ++fill) {
      const int64_t want = std::max<int64_t>(1, std::min(most, fill * 256 / tiles));
      int64_t chunk = (K + want - 1) / want;
      chunk = (chunk + gemm64::TK - 1) / gemm64::TK * gemm64::TK;
      const int64_t used = std::max<int64_t>(1, (K + chunk - 1) / std::max<int64_t>(chunk, 1));
      const double cost = tile_cycles(t, tiles * used, chunk / gemm64::TK) + double(used * M * N) * (16.0 / 2300.0);
      if (least < 0.0 || cost < least) {
        least = cost;
        best = {t, chunk, int(used)};
      }
    }
  }
  return best;
}

// Sums::chain: the tiles that fill the chip at the mixed tier's products (m x m
// and n x m; bits do not depend on the tile).
template <typename F>
void with_chain_tile(int64_t M, int64_t N, const F& f) {
  if (tiles_of({2, 4}, M, N) >= 256) return f(std::integral_constant<int, 2>(), std::integral_constant<int, 4>());
  return f(std::integral_constant<int, 1>(), std::integral_constant<int, 1>());
}

// Sums::chain: at most 512 workgroups' worth of 64 x 64 tiles and 256 chunks,
// 256 k at least in each.
int64_t chain_chunk(int64_t M, int64_t N, int64_t K) {
  const int64_t tiles = ((M + 63) / 64) * ((N + 63) / 64);
  const int64_t splits = std::min<int64_t>(
      {std::max<int64_t>(1, 512 / tiles), std::max<int64_t>(1, K / 256), int64_t(256)});
  return ((K + splits - 1) / splits + gemm64::TK - 1) / gemm64::TK * gemm64::TK;
}

template <bool TA>
void launch_chain(hipStream_t s, int64_t M, int64_t N, int64_t K, double alpha, const double* A, int64_t lda,
                  const double* B, int64_t ldb, double beta, double* C, int64_t ldc) {
  with_chain_tile(M, N, [&](auto rb, auto nb) {
    constexpr int RB = decltype(rb)::value, NB = decltype(nb)::value;
    const int64_t tiles_n = (N + 16 * NB - 1) / (16 * NB), total = tiles_of({RB, NB}, M, N);
    hipLaunchKernelGGL((gemm64::k_gemm_nn<RB, NB, TA, true>), dim3(xcd_grid(total)), dim3(256), 0, s, M, N, K,
                       int(tiles_n), int(total), alpha, A, lda, B, ldb, beta, C, ldc);
  });
}

void chain_tn(hipStream_t s, int64_t M, int64_t N, int64_t K, double alpha, const double* A, int64_t lda,
              const double* B, int64_t ldb, double beta, double* C, int64_t ldc, double* work) {
  const int64_t chunk = chain_chunk(M, N, K), used = chunk > 0 ? (K + chunk - 1) / chunk : 1;
  if (used <= 1) return launch_chain<true>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
  with_chain_tile(M, N, [&](auto rb, auto nb) {
    constexpr int RB = decltype(rb)::value, NB = decltype(nb)::value;
    const int64_t tiles_m = (M + 64 * RB - 1) / (64 * RB), tiles = tiles_of({RB, NB}, M, N), total = tiles * used;
    hipLaunchKernelGGL((gemm64::k_gemm_tn<RB, NB, true>), dim3(xcd_grid(total)), dim3(256), 0, s, M, N, K, chunk,
                       int(tiles_m), int(tiles), int(total), A, lda, B, ldb, work);
  });
  hipLaunchKernelGGL(gemm64::k_gemm_reduce<true>, dim3(unsigned((M * N + 63) / 64)), dim3(256), 0, s, M, N, int(used),
                     alpha, work, beta, C, ldc);
}
}  // namespace

void gemm_nn(hipStream_t s, int64_t M, int64_t N, int64_t K, double alpha, const double* A, int64_t lda,
             const double* B, int64_t ldb, double beta, double* C, int64_t ldc, Sums sums) {
  if (M <= 0 || N <= 0) return;
  if (sums == Sums::chain) return launch_chain<false>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
  if (short_product(M, N, K)) return launch_short<false>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
  const int64_t slices = (K + gemm64::TK - 1) / gemm64::TK;
  const TileShape* best = &kTiles[0];
  for (const TileShape& t : kTiles)
    if (tile_cycles(t, tiles_of(t, M, N), slices) < tile_cycles(*best, tiles_of(*best, M, N), slices)) best = &t;
  with_tile(*best, [&](auto rb, auto nb) {
    constexpr int RB = decltype(rb)::value, NB = decltype(nb)::value;
    const int64_t tiles_n = (N + 16 * NB - 1) / (16 * NB), total = tiles_of({RB, NB}, M, N);
    hipLaunchKernelGGL((gemm64::k_gemm_nn<RB, NB>), dim3(xcd_grid(total)), dim3(256), 0, s, M, N, K, int(tiles_n),
                       int(total), alpha, A, lda, B, ldb, beta, C, ldc);
  });
}

// Monotone in M, N and K, and never below max_splits M N (nor the chunks of
// Sums::chain: at most 512 of 4096 values, K / 256 M N), so one buffer serves
// every call up to its sizing shape.
int64_t gemm_tn_work(int64_t M, int64_t N, int64_t K) {
  const int64_t few = std::max<int64_t>(1, std::min<int64_t>(K / 256, 8));
  if (K < 1024) return few * M * N;
  return std::min(K / 64 * M * N, std::max(few * M * N, int64_t(1) << 21));
}

void gemm_tn(hipStream_t s, int64_t M, int64_t N, int64_t K, double alpha, const double* A,
             int64_t lda, const double* B, int64_t ldb, double beta, double* C, int64_t ldc,
             double* work, Sums sums) {
  if (M <= 0 || N <= 0) return;
  if (sums == Sums::chain) return chain_tn(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, work);
  if (short_product(M, N, K)) return launch_short<true>(s, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
  const TnPlan p = tn_plan(M, N, K);
  with_tile(p.tile, [&](auto rb, auto nb) {
    constexpr int RB = decltype(rb)::value, NB = decltype(nb)::value;
    const int64_t tiles_m = (M + 64 * RB - 1) / (64 * RB), tiles = tiles_of({RB, NB}, M, N);
    const int64_t total = tiles * p.splits;
    hipLaunchKernelGGL((gemm64::k_gemm_tn<RB, NB>), dim3(xcd_grid(total)), dim3(256), 0, s, M, N, K, p.chunk,
                       int(tiles_m), int(tiles), int(total), A, lda, B, ldb, work);
  });
  hipLaunchKernelGGL(gemm64::k_gemm_reduce<>, dim3(unsigned((M * N + 63) / 64)), dim3(256), 0, s, M, N, p.splits, alpha,
                     work, beta, C, ldc);
}

}  // namespace bd

// ---------------------------------------------------------------------------
// C ABI: the GEMMs as stand-alone entry points (row a28 check and tooling).
// ---------------------------------------------------------------------------
extern "C" int64_t bd_gemm_workspace(int32_t mode, int32_t trans_a, int64_t M, int64_t N, int64_t K) {
  if (!trans_a) return 0;
  return mode == 1 ? bd::gemm_tn_bf16x3_work(M, N, K) : bd::gemm_tn_work(M, N, K);
}

extern "C" bd_status bd_gemm_dev(int32_t mode, int32_t trans_a, int64_t M, int64_t N, int64_t K, double alpha,
                                 const double* A, int64_t lda, const double* B, int64_t ldb, double beta,
                                 double* C, int64_t ldc, double* work) {
  BD_GUARD({
    if (M < 0 || N < 0 || K < 0 || (mode != 0 && mode != 1)) bd::fail(BD_ERR_INVALID_PARAMETER, "gemm shape/mode");
    if (trans_a && !work && M * N > 0) bd::fail(BD_ERR_INVALID_PARAMETER, "gemm workspace");
    bd::Gemm g;
    g.bf16x3 = mode == 1;
    if (trans_a) g.tn(nullptr, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc, work);
    else g.nn(nullptr, M, N, K, alpha, A, lda, B, ldb, beta, C, ldc);
    if (hipDeviceSynchronize() != hipSuccess || hipGetLastError() != hipSuccess)
      bd::fail(BD_ERR_DEVICE, "gemm launch failed");
  });
}

// The same product `reps` times back to back on one stream between two HIP
// events (no host round trip in between): the average milliseconds per
// product in *ms. For measuring the kernels apart from the call overhead.
#define GEMM_HIP(call)                                                               \
  do {                                                                               \
    const hipError_t e_ = (call);                                                    \
    if (e_ != hipSuccess) bd::fail(BD_ERR_DEVICE, std::string(#call) + ": " + hipGetErrorString(e_)); \
  } while (0)

extern "C" bd_status bd_gemm_time_dev(int32_t mode, int32_t trans_a, int64_t M, int64_t N, int64_t K,
                                      const double* A, int64_t lda, const double* B, int64_t ldb, double* C,
                                      int64_t ldc, double* work, int32_t reps, double* ms) {
  BD_GUARD({
    if (M < 0 || N < 0 || K < 0 || (mode != 0 && mode != 1) || reps <= 0 || !ms)
      bd::fail(BD_ERR_INVALID_PARAMETER, "gemm timing shape/mode");
    if (trans_a && !work && M * N > 0) bd::fail(BD_ERR_INVALID_PARAMETER, "gemm workspace");
    bd::Gemm g;
    g.bf16x3 = mode == 1;
    hipStream_t s = nullptr;
    hipEvent_t e0 = nullptr, e1 = nullptr;
    GEMM_HIP(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
    GEMM_HIP(hipEventCreate(&e0));
    GEMM_HIP(hipEventCreate(&e1));
    auto run = [&] {
      if (trans_a) g.tn(s, M, N, K, 1.0, A, lda, B, ldb, 0.0, C, ldc, work);
      else g.nn(s, M, N, K, 1.0, A, lda, B, ldb, 0.0, C, ldc);
    };
    run();
    GEMM_HIP(hipEventRecord(e0, s));
    for (int r = 0; r < reps; ++r) run();
    GEMM_HIP(hipEventRecord(e1, s));
    GEMM_HIP(hipEventSynchronize(e1));
    float t = 0.f;
    GEMM_HIP(hipEventElapsedTime(&t, e0, e1));
    *ms = double(t) / reps;
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipStreamDestroy(s);
  });
}

extern "C" bd_status bd_mfma_f64_probe_dev(const double* a, const double* b, double* d) {
  BD_GUARD({
    if (!a || !b || !d) bd::fail(BD_ERR_INVALID_PARAMETER, "null argument");
    hipLaunchKernelGGL(bd::k_mfma_f64_probe, dim3(1), dim3(64), 0, nullptr, a, b, d);
    if (hipDeviceSynchronize() != hipSuccess) bd::fail(BD_ERR_DEVICE, "probe failed");
  });
}

extern "C" bd_status bd_mfma_probe_dev(const uint16_t* a_bits, const uint16_t* b_bits, float* d) {
  BD_GUARD({
    bd::mfma_probe(nullptr, a_bits, b_bits, d);
    if (hipDeviceSynchronize() != hipSuccess) bd::fail(BD_ERR_DEVICE, "probe failed");
  });
}
