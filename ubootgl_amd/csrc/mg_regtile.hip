// mg_regtile.hip -- the level passes of the single-domain multigrid
// (solveLevel, pressure_solver.cpp:201-248): one launch for pre-smoothing,
// residual and restriction, one for prolongation, correction and
// post-smoothing, one workgroup per tile (tile bodies in
// regtile_device.hpp).
#include "regtile_device.hpp"

namespace ubg {
namespace {

// tile (X0, Y0) of an otx x oty partition, blocks in XCD-grouped order
__device__ __forceinline__ void tile_origin(int ntx, int otx, int oty, int &X0, int &Y0) {
  const int b = xcd_tile(blockIdx.x, gridDim.x);
  X0 = (b % ntx) * otx;
  Y0 = (b / ntx) * oty;
}

template <class T, bool ZP, bool ZG>
__global__ void __launch_bounds__(T::TPB, T::MINW)
    k_level_pre(const float *__restrict__ p, float *__restrict__ p_out,
                const float *__restrict__ f, const uint8_t *__restrict__ m, int w, int h,
                float hh, float alpha, float ihsq, float *__restrict__ fc,
                float *__restrict__ ec, int wc, int hc, int otx, int oty, int ntx) {
  extern __shared__ __align__(16) char smem[];
  int X0, Y0;
  tile_origin(ntx, otx, oty, X0, Y0);
  regtile_pre<T, ZP, ZG>(smem, X0, Y0, otx, oty, p, p_out, f, m, w, h, hh, alpha, ihsq, fc, ec,
                         wc, hc);
}

template <class T, bool ZG>
__global__ void __launch_bounds__(T::TPB, T::MINW)
    k_level_post(const float *__restrict__ p, float *__restrict__ p_out,
                 const float *__restrict__ f, const uint8_t *__restrict__ m, int w, int h,
                 float hh, float alpha, const float *__restrict__ ec,
                 const uint8_t *__restrict__ mc, int wc, int hc, int otx, int oty, int ntx) {
  extern __shared__ __align__(16) char smem[];
  int X0, Y0;
  tile_origin(ntx, otx, oty, X0, Y0);
  regtile_post<T, ZG>(smem, X0, Y0, otx, oty, p, p_out, f, m, w, h, hh, alpha, ec, mc, wc, hc);
}

// n cells in tiles of at most `most` (even), evenly split: k tiles of o cells
void split(int n, int most, int &o, int &k) {
  k = (n + most - 1) / most;
  o = ((n + k - 1) / k + 1) & ~1;
  k = (n + o - 1) / o;
}

long tiles(const Level &L, PassShape shape, bool pre, int nu) {
  int otx, oty;
  pass_tile(shape, pre, nu, &otx, &oty);
  return (long)((L.w + otx - 1) / otx) * ((L.h + oty - 1) / oty);
}
// fn(the level's RegTile).  Beyond the shapes of pass_shape: three sweeps on
// more than 32 tiles per CU take 12 waves of 6 rows, whose halo is an even
// smaller share.  Both compiled for 6 waves a SIMD, pre + post in us with 12
// waves against 8, under the zero-gradient BC and without it:
//   8192x4096  152 + 138 against 168 + 144    147 + 133 against 162 + 132
//   6144x3072   77 +  79 against  83 +  82     73 +  76 against  78 +  74
//   4096x2048   41 +  39 against  42 +  40     37 +  35 against  39 +  37
//   3072x1536   30 +  27 against  29 +  28     27 +  25 against  27 +  25
//   2048x1024   19 +  18 against  18 +  18     16 +  17 against  16 +  17
// 4096x2048 (18 tiles per CU) stays with 8: a whole step (627 us) and a whole
// solve (8.73 ms) there take the same with either, within 0.5%.  With two sweeps the post pass loses, 129
// against 122 at 8192x4096, and the pre pass gains as much.
template <class Fn> void with_level(const Level &L, bool pre, int nu, Fn fn) {
  const long small = tiles(L, PASS_SMALL, pre, nu);
  if (nu == 3 && small > 32 * kPassCUs) fn(RegTile<3, 6, 12>{});
  else with_pass(pass_shape(tiles(L, PASS_TINY, pre, nu), small), nu, fn);
}

void swap_p(Level &L) {
  float *t = L.p;
  L.p = L.p_alt;
  L.p_alt = t;
}

} // namespace

void launch_level_pre(Level &L, Level &C, int nu, float h, float alpha, bool zero_p, bool zg,
                      bool zero_coarse, hipStream_t s) {
  with_level(L, true, nu, [&](auto t) {
    using T = decltype(t);
    int otx, ntx, oty, nty;
    split(L.w, T::OTXP, otx, ntx);
    split(L.h, T::OTYP, oty, nty);
    auto k = zero_p ? k_level_pre<T, true, false>
                    : (zg ? k_level_pre<T, false, true> : k_level_pre<T, false, false>);
    launch_k(k, dim3(ntx * nty), dim3(T::TPB), (uint32_t)T::LDS, s, L.p, L.p_alt, L.f, L.mask, L.w,
             L.h, h, alpha, 1.0f / h / h, C.f, zero_coarse ? C.p : nullptr, C.w, C.h, otx, oty,
             ntx);
  });
  swap_p(L);
}

void launch_level_post(Level &L, const Level &C, int nu, float h, float alpha, bool zg,
                       hipStream_t s) {
  with_level(L, false, nu, [&](auto t) {
    using T = decltype(t);
    int otx, ntx, oty, nty;
    split(L.w, T::OTXQ, otx, ntx);
    split(L.h, T::OTYQ, oty, nty);
    launch_k(zg ? k_level_post<T, true> : k_level_post<T, false>, dim3(ntx * nty), dim3(T::TPB),
             (uint32_t)T::LDS, s, L.p, L.p_alt, L.f, L.mask, L.w, L.h, h, alpha, C.p, C.mask, C.w,
             C.h, otx, oty, ntx);
  });
  swap_p(L);
}

} // namespace ubg
