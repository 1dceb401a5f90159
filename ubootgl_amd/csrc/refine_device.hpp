// refine_device.hpp -- the float64 refinement update as a device function over
// one column of kIrRows rows (a block: 256 columns), shared by the single
// solve and the batched one, whose sums of r^2 are then the same.
#pragma once

#include "mg_device.hpp"

namespace ubg {

constexpr int kIrCols = 256, kIrRows = 8;

// the lane to the left's / right's value
__device__ __forceinline__ double left_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x138, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x138, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double right_f64(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x130, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x130, 0xf, 0xf, true);
  return __hiloint2double(hi, lo);
}

// x_b = x_a + e (ACC) or x_a, r32 = (float) r(x_b), e_zero = 0 in column x,
// rows y0 .. y0 + kIrRows - 1; returns the column's sum of r^2, rows in order.
// Neighbour values x_a(n) + e(n) are formed from the inputs, so no thread
// reads a value another thread writes.  Every thread of the wave takes part
// (columns beyond w store nothing): the values left and right of a column
// come from the lanes next to it, and the wave's first and last lane load
// theirs.
//
// Bound by memory on large grids (33 bytes a cell) and by latency on small
// ones, so all loads of the 8 rows are issued before the first use: 8192x4096
// 188 us (5.9 TB/s) and 1024x512 7.1 us, where loading a neighbour only after
// its mask bit, row by row, took 297 and 13.4.
template <bool ACC>
__device__ __forceinline__ double
ir_update_column(int x, int y0, const double *__restrict__ xa, double *__restrict__ xb,
                 const float *__restrict__ e, float *__restrict__ ez,
                 const float *__restrict__ f, const uint8_t *__restrict__ m,
                 float *__restrict__ r32, int w, int h, double ihsq) {
  constexpr int R = kIrRows;
  const int lane = threadIdx.x & 63, xc = min(x, w - 1);
  const bool side = lane == 0 || lane == 63;
  const int xs = lane == 0 ? max(xc - 1, 0) : min(xc + 1, w - 1);
  double X[R + 2], S[R];
  float E[R + 2], ES[R], fv[R];
  unsigned mk[R];
  auto row = [&](int j) { return (size_t)min(max(y0 + j, 0), h - 1) * w; };
#pragma unroll
  for (int j = 0; j < R + 2; j++) {
    X[j] = xa[row(j - 1) + xc];
    if (ACC) E[j] = e[row(j - 1) + xc];
  }
#pragma unroll
  for (int j = 0; j < R; j++) {
    mk[j] = m[row(j) + xc];
    fv[j] = f[row(j) + xc];
    S[j] = 0.0;
    ES[j] = 0.0f;
  }
  if (side) {
#pragma unroll
    for (int j = 0; j < R; j++) {
      S[j] = xa[row(j) + xs];
      if (ACC) ES[j] = e[row(j) + xs];
    }
  }
  if (ACC) {
#pragma unroll
    for (int j = 0; j < R + 2; j++) X[j] += (double)E[j];
#pragma unroll
    for (int j = 0; j < R; j++) S[j] += (double)ES[j];
  }
  const bool inx = x >= 1 && x <= w - 2;
  double acc = 0.0;
#pragma unroll
  for (int j = 0; j < R; j++) {
    const int y = y0 + j;
    if (y >= h) break;
    const double c = X[j + 1];
    double l = left_f64(c), r = right_f64(c);
    l = lane == 0 ? S[j] : l;
    r = lane == 63 ? S[j] : r;
    double s = 0.0;
    s = mk[j] & MK_W ? s + (l - c) : s;
    s = mk[j] & MK_E ? s + (r - c) : s;
    s = mk[j] & MK_S ? s + (X[j] - c) : s;
    s = mk[j] & MK_N ? s + (X[j + 2] - c) : s;
    double res = (double)fv[j] + s * ihsq;
    res = inx && y >= 1 && y <= h - 2 && (mk[j] & MK_SELF) ? res : 0.0;
    if (x < w) {
      const size_t i = (size_t)y * w + x;
      xb[i] = c;
      ez[i] = 0.0f;
      r32[i] = (float)res;
      acc += res * res;
    }
  }
  return acc;
}

// a thread's share of n partial sums in a block of 1024 threads (every
// 1024th, in order), eight loads in flight
__device__ __forceinline__ double thread_partials(const double *__restrict__ p, int n) {
  double s = 0.0;
  for (int b = threadIdx.x; b < n; b += 8 * 1024) {
    double v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = p[min(b + 1024 * k, n - 1)];
#pragma unroll
    for (int k = 0; k < 8; k++)
      if (b + 1024 * k < n) s += v[k];
  }
  return s;
}

} // namespace ubg
