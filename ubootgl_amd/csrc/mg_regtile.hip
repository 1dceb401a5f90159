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
__global__ void __launch_bounds__(T::TPB, 4)
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
__global__ void __launch_bounds__(T::TPB, 4)
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

template <class T> struct PreLaunch {
  static void run(Level &L, Level &C, float h, float alpha, bool zero_p, bool zg,
                  bool zero_coarse, hipStream_t s) {
    int otx, ntx, oty, nty;
    split(L.w, T::OTXP, otx, ntx);
    split(L.h, T::OTYP, oty, nty);
    const float ihsq = 1.0f / h / h;
    auto k = zero_p ? (zg ? k_level_pre<T, true, true> : k_level_pre<T, true, false>)
                    : (zg ? k_level_pre<T, false, true> : k_level_pre<T, false, false>);
    launch_k(k, dim3(ntx * nty), dim3(T::TPB), (uint32_t)T::LDS, s, L.p, L.p_alt, L.f, L.mask, L.w,
             L.h, h, alpha, ihsq, C.f, zero_coarse ? C.p : nullptr, C.w, C.h, otx, oty, ntx);
  }
};

template <class T> struct PostLaunch {
  static void run(Level &L, const Level &C, float h, float alpha, bool zg, hipStream_t s) {
    int otx, ntx, oty, nty;
    split(L.w, T::OTXQ, otx, ntx);
    split(L.h, T::OTYQ, oty, nty);
    launch_k(zg ? k_level_post<T, true> : k_level_post<T, false>, dim3(ntx * nty), dim3(T::TPB),
             (uint32_t)T::LDS, s, L.p, L.p_alt, L.f, L.mask, L.w, L.h, h, alpha, C.p, C.mask, C.w,
             C.h, otx, oty, ntx);
  }
};

// Tile shape by the number of 128 x 32 regions a level's pre pass splits
// into.  Up to one per CU: 16 waves of 2 rows, the least work per wave and
// phase, since such a launch is all latency (512x256 at 2/2: 5.2 + 5.4 us
// against 6.0 + 6.7 us with 8 waves of 4 rows).  Up to four: 8 waves of 4
// rows, so that several workgroups share a CU and one loads while another
// computes (1280x720 at 3/3: 10.4 + 10.0 us against 11.3 + 11.4 us with 8
// waves of 6 rows and 11.1 + 9.7 us with 16 of 2).  Above: 8 waves of 6 rows,
// whose halo rows are a smaller share (4096x2048 at 2/2: 33.6 + 31.2 us
// against 38.5 + 35.5 us with 8 rows, whose fewer workgroups overlap less;
// 3072x1536 at 3/3: 29.2 + 27.0 us against 32.6 + 28.9 us with 4).
template <int NU, template <class> class Launch, typename... Args>
void launch_shape(const Level &L, Args &&...args) {
  using Small = RegTileSmall<NU>;
  using Mid = RegTileMid<NU>;
  using Big = RegTileBig<NU>;
  const long tiles = (long)((L.w + Small::OTXP - 1) / Small::OTXP) *
                     ((L.h + Small::OTYP - 1) / Small::OTYP);
  if (tiles <= 256) Launch<Small>::run(args...);
  else if (tiles <= 1024) Launch<Mid>::run(args...);
  else Launch<Big>::run(args...);
}

template <template <class> class Launch, typename... Args>
void launch_nu(int nu, const Level &L, Args &&...args) {
  switch (nu) {
  case 0: launch_shape<0, Launch>(L, args...); break;
  case 1: launch_shape<1, Launch>(L, args...); break;
  case 2: launch_shape<2, Launch>(L, args...); break;
  default: launch_shape<3, Launch>(L, args...); break;
  }
}

void swap_p(Level &L) {
  float *t = L.p;
  L.p = L.p_alt;
  L.p_alt = t;
}

} // namespace

void launch_level_pre(Level &L, Level &C, int nu, float h, float alpha, bool zero_p, bool zg,
                      bool zero_coarse, hipStream_t s) {
  launch_nu<PreLaunch>(nu, L, L, C, h, alpha, zero_p, zg, zero_coarse, s);
  swap_p(L);
}

void launch_level_post(Level &L, const Level &C, int nu, float h, float alpha, bool zg,
                       hipStream_t s) {
  launch_nu<PostLaunch>(nu, L, L, C, h, alpha, zg, s);
  swap_p(L);
}

} // namespace ubg
