// The paired plane pass: shapes and launches (the kernels are in
// plane_kernels.hpp, one source per type and mode).
#include "plane.hpp"

#include <algorithm>
#include <string>

#include "common.hpp"

namespace bd {
namespace {

constexpr int kLds = 160 * 1024;

template <typename F>
const void* kernel_of(const PairShape& s, int mode) {
  const int n1 = s.split * s.ny;
  return mode == 0   ? pair_kernel<F, 0>(s.split, n1, s.n2)
         : mode == 1 ? pair_kernel<F, 1>(s.split, n1, s.n2)
                     : pair_kernel<F, 2>(s.split, n1, s.n2);
}

}  // namespace

PairShape pair_shape(int n1, int n2, int Z, size_t elem) {
  PairShape s;
  double best = 0.0;
  for (int split : {1, 2}) {
    PlaneLayout l;
    if (!plane_layout(split, n1, n2, l)) continue;
    const int chunks = (n1 / split + l.rows - 1) / l.rows;
    for (int waves = 8; waves >= 2; --waves) {
      const size_t lds = size_t(Z * l.ldp + n1 + n2) * elem + size_t(waves) * l.words * (elem / 2);
      if (lds > kLds) continue;
      // Wavefronts in flight on a CU, less those idle in the last round of z
      // rows. 72^2 FP64, 80 pairs: 6 wavefronts (12 a CU).
      const double fill = double(chunks) / (waves * ((chunks + waves - 1) / waves));
      const int per_simd = elem == 16 ? l.simd_f64 : l.simd_f32;
      const double score = fill * std::min<int>(4 * per_simd, int(kLds / lds) * waves);
      // By row parity only where whole planes leave a CU under 6 wavefronts:
      // it reads the sticks twice.
      if (score > best && !(split == 2 && best >= 5.0)) {
        best = score;
        s.on = true;
        s.split = split;
        s.ny = n1 / split;
        s.n2 = n2;
        s.waves = waves;
        s.lds = lds;
      }
    }
  }
  return s;
}

template <typename F>
void pair_allow_lds(const PairShape& s) {
  if (!s.on) return;
  for (int mode : {0, 1, 2}) {
    const hipError_t e =
        hipFuncSetAttribute(kernel_of<F>(s, mode), hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
    if (e != hipSuccess) fail(BD_ERR_DEVICE, std::string("plane kernel LDS: ") + hipGetErrorString(e));
  }
}

template <typename F>
void pair_launch(hipStream_t s, const PairShape& shape, int mode, const PairArgs<F>& a, int groups) {
  const dim3 grid = mode == 1 ? dim3(unsigned(a.n0), unsigned(groups)) : dim3(unsigned(a.pairs), unsigned(a.n0));
  PairArgs<F> args = a;
  void* params[] = {&args};
  const hipError_t e =
      hipLaunchKernel(kernel_of<F>(shape, mode), grid, dim3(64 * shape.waves), params, shape.lds, s);
  if (e != hipSuccess) fail(BD_ERR_DEVICE, std::string("plane launch: ") + hipGetErrorString(e));
}

template void pair_allow_lds<double>(const PairShape&);
template void pair_allow_lds<float>(const PairShape&);
template void pair_launch<double>(hipStream_t, const PairShape&, int, const PairArgs<double>&, int);
template void pair_launch<float>(hipStream_t, const PairShape&, int, const PairArgs<float>&, int);

}  // namespace bd
