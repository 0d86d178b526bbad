// The paired plane pass: y and z transforms of one y-z plane as two in-register
// radix passes per line (plane_kernels.hpp).
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "fft_device.hpp"

namespace bd {

// One z line of the occupied sticks: its sticks sit at positions
// first, first + 1, ... of the stick buffer, for y = start, start + 1, ...
// (mod n1), count of them.
struct PlaneLine {
  int first, start, count, pad;
};

// Arguments of the kernels.
template <typename F>
struct PairArgs {
  const c2<F>* in;          // sticks [pair][x][Spad]
  c2<F>* out;               // the same layout (may be `in` when split == 1)
  const PlaneLine* lines;   // Z, cyclically from z = zs
  const c2<double>* roots;  // [n0 | n1 | n2]
  const F* potential;       // V (or dV), full grid
  const c2<F>* kept_in;     // mode 2: real-space pair fields
  c2<F>* kept_out;          // mode 1: written when not null
  const double* weights;    // mode 1: two per pair
  double* rho;              // mode 1: partial densities, one grid per group
  double inv_volume;
  int n0, Spad, Z, zs, pairs;
};

// What the host needs to know of a kernel: LDS row of a line (complex
// values), exchange words and z rows of a wavefront, wavefronts per SIMD its
// registers allow.
struct PlaneLayout {
  int ldp, words, rows, simd_f64, simd_f32;
};
// false: no kernel for this plane.
bool plane_layout(int split, int n1, int n2, PlaneLayout& out);
template <typename F, int MODE>
const void* pair_kernel(int split, int n1, int n2);

// Launch shape of the pass on one plan.
struct PairShape {
  bool on = false;
  int split = 1;  // 1: whole planes; 2: even, then odd y rows
  int ny = 0, n2 = 0;  // rows per pass (n1 / split), z length
  int waves = 0;  // wavefronts per workgroup
  size_t lds = 0;
};
// The shape for Z lines of an n1 x n2 plane, elem = sizeof(c2<F>); off where no
// kernel is built for the plane or it does not fit a workgroup.
PairShape pair_shape(int n1, int n2, int Z, size_t elem);
// Raise the kernels' LDS limit (once per op).
template <typename F>
void pair_allow_lds(const PairShape& s);
// mode 0: sticks -> V psi -> sticks. mode 1: band density into `groups`
// partial grids. mode 2: kept fields -> dV psi -> sticks.
template <typename F>
void pair_launch(hipStream_t s, const PairShape& shape, int mode, const PairArgs<F>& a, int groups);

}  // namespace bd
