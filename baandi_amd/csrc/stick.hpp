// The x pass: columns (ORC rows at Gamma, interleaved Re and Im at k) <->
// x-transformed sticks, each stick as two in-register radix passes of one
// wavefront (stick.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

#include "fft_device.hpp"

namespace bd {

// How a line of n0 = a * b points is cut: sticks per wavefront and per
// workgroup (4 wavefronts), LDS row of a stick (complex values).
struct StickShape {
  bool on = false;
  int a = 0, b = 0, per = 0, tile = 0, row = 0;
};
// off where no kernel is built for the length.
StickShape stick_shape(int n0);

// Arguments of the kernels. `tile` sticks a workgroup; the sticks of a mirror
// unit (+G and -G of its representatives) share a tile.
template <typename F>
struct StickArgs {
  const double* x;
  int64_t ldx;
  double* y;  // forward only
  int64_t ldy;
  int m;              // columns
  int n0, Spad, tiles, pairs;
  int by_xcd;         // deal whole pairs to the XCDs
  const int* rep_at;  // inverse: [tile][wave][r][lane], 0 or +-(representative + 1), at k coefficient + 1
  const int* tile_off;
  const int4* entries;  // forward: (representative, +G, -G positions in the LDS image, 0); at k (coefficient, position, -1, 0)
  const int* dst;       // stick buffer position of each slot
  const c2<double>* roots;
  const double* kinetic;
  double inv_n;
  c2<F>* sticks;  // [pair][x][Spad]
};
// k: one complex column per FFT slot instead of a pair of real ones.
template <typename F>
void stick_inverse(hipStream_t s, const StickShape& shape, StickArgs<F> a, bool k);
// h: y = local part + T_G x; add: y += the local part alone; k: as h, on
// complex columns.
enum class StickOut { h, add, k };
template <typename F>
void stick_forward(hipStream_t s, const StickShape& shape, StickArgs<F> a, StickOut out);

}  // namespace bd
