// batch_level.hip -- the batched solver's level passes (batch_stage.hpp): the
// register tiles of regtile_device.hpp over every member domain's tiles in
// one launch.
#include "batch_stage.hpp"
#include "regtile_device.hpp"

namespace ubg {
namespace {

template <class T, bool ZP, bool ZG>
__global__ void __launch_bounds__(T::TPB, 4) kb_level_pre(StageArgs a) {
  extern __shared__ __align__(16) char smem[];
  TileWalk tw;
  if (!tw.init(a)) return;
  do {
    const BDom &D = a.dom[tw.d];
    if (!dom_active(D)) continue;
    const BLev &F = a.lev[tw.d * BMAXL + a.level];
    const BLev &C = a.lev[tw.d * BMAXL + a.level + 1];
    const int s = a.ia[tw.d];
    __syncthreads(); // the previous tile's LDS readers are done
    // the coarse level's next pass does not read its p: nothing to zero
    regtile_pre<T, ZP, ZG>(smem, tw.tx() * tw.otx, tw.ty() * a.oty, tw.otx, a.oty, F.p[s],
                           F.p[s ^ 1], F.f, F.mask, F.w, F.h, F.hh, a.alpha, F.ihsq, C.f, nullptr,
                           C.w, C.h);
  } while (tw.next(a));
}

template <class T, bool ZG>
__global__ void __launch_bounds__(T::TPB, 4) kb_level_post(StageArgs a) {
  extern __shared__ __align__(16) char smem[];
  TileWalk tw;
  if (!tw.init(a)) return;
  do {
    const BDom &D = a.dom[tw.d];
    if (!dom_active(D)) continue;
    const BLev &F = a.lev[tw.d * BMAXL + a.level];
    const BLev &C = a.lev[tw.d * BMAXL + a.level + 1];
    const int s = a.ia[tw.d];
    __syncthreads();
    regtile_post<T, ZG>(smem, tw.tx() * tw.otx, tw.ty() * a.oty, tw.otx, a.oty, F.p[s], F.p[s ^ 1],
                        F.f, F.mask, F.w, F.h, F.hh, a.alpha, C.p[a.ib[tw.d]], C.mask, C.w, C.h);
  } while (tw.next(a));
}

template <class T>
void launch(bool pre, bool zg, int blocks, hipStream_t s, const StageArgs &a) {
  const bool z = zg && a.level == 0;
  auto k = pre ? (a.level > 0 ? kb_level_pre<T, true, false>
                              : (z ? kb_level_pre<T, false, true> : kb_level_pre<T, false, false>))
               : (z ? kb_level_post<T, true> : kb_level_post<T, false>);
  hipLaunchKernelGGL(k, dim3(blocks), dim3(T::TPB), T::LDS, s, a);
}

} // namespace

void launch_batch_pass(PassShape shape, bool pre, int nu, bool zg, int blocks, hipStream_t s,
                       const StageArgs &a) {
  with_pass(shape, nu, [&](auto t) { launch<decltype(t)>(pre, zg, blocks, s, a); });
}

} // namespace ubg
