// batch_stage.hpp -- internal to the batched solver: what a stage's kernel
// gets, and its walk over the tiles of every member domain.
#pragma once

#include "batch_engine.hpp"

namespace ubg {

struct StageArgs {
  const BLev *lev;
  const BDom *dom;
  const int *off; // tile prefix over domain slots [ndom + 1], tiles per row [ndom], tile width [ndom]
  int ndom;
  int ntiles;
  int level;
  const uint8_t *ia; // per-domain index row a
  const uint8_t *ib; // per-domain index row b
  float alpha;
  int oty; // tile rows of the level passes (their widths are per domain)
};

__device__ __forceinline__ bool dom_active(const BDom &D) {
  return __builtin_amdgcn_readfirstlane(D.st->active) != 0;
}

// Tiles of a stage are split into equal contiguous chunks, one per block of
// the (persistent) grid, in XCD-grouped block order so that neighbouring
// chunks share an XCD's L2.  A block locates the domain slot of its first tile
// once (the last d with off[d] <= t; domains without tiles at this level
// have off[d] == off[d+1]) and then walks forward.
struct TileWalk {
  int t, t1; // current tile, end of the chunk
  int d, j;  // domain slot, tile index within the domain
  int nt, ntx, otx;
  __device__ __forceinline__ bool init(const StageArgs &a) {
    const int per = (a.ntiles + gridDim.x - 1) / gridDim.x;
    const int b = xcd_tile(blockIdx.x, gridDim.x);
    t = b * per;
    t1 = min(t + per, a.ntiles);
    if (t >= t1) return false;
    int lo = 0, hi = a.ndom;
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (a.off[mid] <= t) lo = mid;
      else hi = mid;
    }
    d = lo;
    j = t - a.off[d];
    nt = a.off[d + 1] - a.off[d];
    ntx = a.off[a.ndom + 1 + d];
    otx = a.off[2 * a.ndom + 1 + d];
    return true;
  }
  __device__ __forceinline__ bool next(const StageArgs &a) {
    if (++t >= t1) return false;
    if (++j == nt) {
      do {
        d++;
      } while (a.off[d + 1] == a.off[d]);
      j = 0;
      nt = a.off[d + 1] - a.off[d];
      ntx = a.off[a.ndom + 1 + d];
      otx = a.off[2 * a.ndom + 1 + d];
    }
    return true;
  }
  __device__ __forceinline__ int tx() const { return j % ntx; }
  __device__ __forceinline__ int ty() const { return j / ntx; }
};

// The level passes (mg_regtile.hip's tiles, regtile_device.hpp) over the tiles
// of every member domain at one level, walked as the other stages: pre reads
// p[ia], writes p[ia^1] and the coarse rhs; post reads p[ia] and the coarse
// solution p[ib], writes p[ia^1].  Level 0 reads its p and, with zg, takes
// setZeroGradientBC; the levels below start from zero.
void launch_batch_pass(PassShape shape, bool pre, int nu, bool zg, int blocks, hipStream_t s,
                       const StageArgs &a);

} // namespace ubg
