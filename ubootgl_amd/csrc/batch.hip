// batch.hip -- batched refinement solves (ubg_batch_*): many independent
// domains of uneven size, one launch per multigrid stage.
//
// Per refinement step and domain the arithmetic is exactly that of
// ubg_mg_ir_solve (refine.hip) around MG::solve (pressure_solver.cpp:201-248):
// nu_pre rbgs sweeps (pressure_solver.cpp:49-89), residual + restriction
// (:91-132), the coarse levels from the first one that fits in LDS (one
// workgroup per domain), prolongation + correction (:134-181), nu_post
// sweeps; then the fused float64 update x += e, r = f + A x, and the norm of
// r summed in the single-domain order.  Stages of all domains share one
// launch: a kernel walks a tile list (domain, tile origin) with a fixed grid
// (persistent loop), and reads per-domain buffer indices from a small table
// row of the stage, so domains with different level counts and ping-pong
// parities run in the same launch.  Domains whose solve has ended are
// skipped on the device; no host round trip is needed per stage.
#include "batch_stage.hpp"
#include "mg_device.hpp"
#include "refine_device.hpp"

#include <algorithm>
#include <array>
#include <cstdio>
#include <fstream>
#include <sstream>

namespace ubg {

// ===========================================================================
// kernels
// ===========================================================================
namespace {

constexpr int TPB = 256;

// One red+black rbgs sweep of a TX x TY tile, ping-pong (read p[a], write
// p[a^1]).  p is staged with a 2-cell halo; red cells ((x+y) odd) of the tile
// and a 1-cell ring are updated in LDS from old black values, then black
// cells of the tile from the new red values -- the two-pass order of
// pressure_solver.cpp:65-71, bit for bit.
template <int TX, int TY>
__global__ void __launch_bounds__(TPB) kb_sweep(StageArgs a) {
  static_assert(TX % 2 == 0, "pairs need an even tile width");
  constexpr int PX = TX + 4, PY = TY + 4, RX = TX + 2, RY = TY + 2;
  __shared__ float sp[PY * PX];
  TileWalk tw;
  if (!tw.init(a)) return;
  do {
    const Tile T{tw.d, tw.tx() * TX, tw.ty() * TY, tw.j};
    const BDom &D = a.dom[T.d];
    if (!dom_active(D)) continue;
    const BLev &L = a.lev[T.d * BMAXL + a.level];
    const int s = a.ia[T.d];
    const float *__restrict__ src = L.p[s];
    float *__restrict__ dst = L.p[s ^ 1];
    const float *__restrict__ fv = L.f;
    const uint8_t *__restrict__ mk = L.mask;
    const int w = L.w, h = L.h;
    const float hh = L.hh;
    __syncthreads(); // the previous tile's readers are done with sp
    for (int i = threadIdx.x; i < PX * PY; i += TPB) {
      const int r = i / PX, c = i - r * PX;
      const int gx = T.x0 - 2 + c, gy = T.y0 - 2 + r;
      sp[i] = (gx >= 0 && gx < w && gy >= 0 && gy < h) ? src[(size_t)gy * w + gx] : 0.0f;
    }
    __syncthreads();
    // red: one red cell per horizontal pair (columns x0-1+2q, x0+2q)
    for (int i = threadIdx.x; i < RY * (RX / 2); i += TPB) {
      const int r = i / (RX / 2), q = i - r * (RX / 2);
      const int gy = T.y0 - 1 + r;
      const int c0 = T.x0 - 1 + 2 * q;
      const int gx = ((c0 + gy) & 1) ? c0 : c0 + 1;
      if (gx >= 1 && gx <= w - 2 && gy >= 1 && gy <= h - 2) {
        const size_t gi = (size_t)gy * w + gx;
        const int li = (r + 1) * PX + (gx - T.x0 + 2);
        sp[li] = smooth(sp[li], sp[li - 1], sp[li + 1], sp[li - PX], sp[li + PX], fv[gi], mk[gi],
                        hh, a.alpha);
      }
    }
    __syncthreads();
    // black: one black cell per pair (columns x0+2q, x0+2q+1); both cells of
    // the pair are stored
    for (int i = threadIdx.x; i < TY * (TX / 2); i += TPB) {
      const int r = i / (TX / 2), q = i - r * (TX / 2);
      const int gy = T.y0 + r;
      if (gy >= h) continue;
      const int c0 = T.x0 + 2 * q;
      const int li0 = (r + 2) * PX + 2 * q + 2;
      float v0 = sp[li0], v1 = sp[li0 + 1];
      const int bx = ((c0 + gy) & 1) ? c0 + 1 : c0; // the black one
      if (bx < w && bx >= 1 && bx <= w - 2 && gy >= 1 && gy <= h - 2) {
        const size_t gi = (size_t)gy * w + bx;
        const int li = li0 + (bx - c0);
        const float nb = smooth(sp[li], sp[li - 1], sp[li + 1], sp[li - PX], sp[li + PX], fv[gi],
                                mk[gi], hh, a.alpha);
        if (bx == c0) v0 = nb;
        else v1 = nb;
      }
      const size_t g0 = (size_t)gy * w + c0;
      if (c0 < w) dst[g0] = v0;
      if (c0 + 1 < w) dst[g0 + 1] = v1;
    }
  } while (tw.next(a));
}

// calculateResidualField + restrict (pressure_solver.cpp:91-132) for a tile
// of 32 x 8 interior coarse cells; the coarse solution is zeroed (:224).
// ia: fine p index, ib: coarse p index.
constexpr int RCX = 32, RCY = 8, RFX = 2 * RCX + 1, RFY = 2 * RCY + 1, RPX = RFX + 2,
              RPY = RFY + 2;
__global__ void __launch_bounds__(TPB) kb_rr(StageArgs a) {
  __shared__ float sp[RPY][RPX];
  __shared__ float sr[RFY][RFX + 1];
  TileWalk tw;
  if (!tw.init(a)) return;
  do {
    const Tile T{tw.d, 1 + tw.tx() * RCX, 1 + tw.ty() * RCY, tw.j};
    const BDom &D = a.dom[T.d];
    if (!dom_active(D)) continue;
    const BLev &F = a.lev[T.d * BMAXL + a.level];
    const BLev &C = a.lev[T.d * BMAXL + a.level + 1];
    const float *__restrict__ p = F.p[a.ia[T.d]];
    const int wf = F.w, hf = F.h, wc = C.w, hc = C.h;
    const int fx0 = 2 * T.x0 - 1, fy0 = 2 * T.y0 - 1; // residual region origin
    __syncthreads();
    for (int i = threadIdx.x; i < RPX * RPY; i += TPB) {
      const int r = i / RPX, c = i - r * RPX;
      const int gx = fx0 - 1 + c, gy = fy0 - 1 + r;
      (&sp[0][0])[i] = (gx >= 0 && gx < wf && gy >= 0 && gy < hf) ? p[(size_t)gy * wf + gx] : 0.0f;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < RFX * RFY; i += TPB) {
      const int r = i / RFX, c = i - r * RFX;
      const int gx = fx0 + c, gy = fy0 + r;
      float res = 0.0f;
      if (gx >= 1 && gx < wf - 1 && gy >= 1 && gy < hf - 1) {
        const size_t gi = (size_t)gy * wf + gx;
        res = residual_of(sp[r + 1][c + 1], sp[r + 1][c], sp[r + 1][c + 2], sp[r][c + 1],
                          sp[r + 2][c + 1], F.f[gi], F.mask[gi], F.ihsq);
      }
      sr[r][c] = res;
    }
    __syncthreads();
    const int cx = threadIdx.x % RCX, cy = threadIdx.x / RCX;
    const int X = T.x0 + cx, Y = T.y0 + cy;
    if (X < wc - 1 && Y < hc - 1) {
      const int r = 2 * cy + 1, c = 2 * cx + 1;
      auto R = [&](int dx, int dy) { return sr[r + dy][c + dx]; };
      float vv = 0.0f;
      vv = R(-1, -1) * 1.0f + R(0, -1) * 2.0f + R(1, -1) * 1.0f;
      vv += R(-1, 0) * 2.0f + R(0, 0) * 4.0f + R(1, 0) * 2.0f;
      vv += R(-1, 1) * 1.0f + R(0, 1) * 2.0f + R(1, 1) * 1.0f;
      const size_t ci = (size_t)Y * wc + X;
      C.f[ci] = vv * (1.0f / 16.0f);
      C.p[a.ib[T.d]][ci] = 0.0f;
    }
  } while (tw.next(a));
}

// prolongate + correct (pressure_solver.cpp:134-181) for a tile of 256 x 8
// interior fine cells (one column per thread), in place on p[ia]; the coarse
// solution is p[ib] of the next level.
constexpr int PCW = 256, PCH = 8;
__global__ void __launch_bounds__(TPB) kb_pc(StageArgs a) {
  TileWalk tw;
  if (!tw.init(a)) return;
  do {
    const Tile T{tw.d, 1 + tw.tx() * PCW, 1 + tw.ty() * PCH, tw.j};
    const BDom &D = a.dom[T.d];
    if (!dom_active(D)) continue;
    const BLev &F = a.lev[T.d * BMAXL + a.level];
    const BLev &C = a.lev[T.d * BMAXL + a.level + 1];
    const int w = F.w, h = F.h, wc = C.w;
    const int x = T.x0 + threadIdx.x;
    if (x >= w - 1) continue;
    float *__restrict__ p = F.p[a.ia[T.d]];
    const float *__restrict__ ec = C.p[a.ib[T.d]];
    const uint8_t *__restrict__ mc = C.mask;
    const int ax = x >> 1;
    const bool xe = !(x & 1);
    auto E = [&](int xx, int yy) { return ec[(size_t)yy * wc + xx]; };
    auto FC = [&](int xx, int yy) { return (int)(mc[(size_t)yy * wc + xx] & MK_SELF); };
    const int y1 = min(T.y0 + PCH, h - 1);
    for (int y = T.y0; y < y1; y++) {
      const size_t i = (size_t)y * w + x;
      const float Fv = (F.mask[i] & MK_SELF) ? 1.0f : 0.0f;
      const int by = y >> 1;
      const bool ye = !(y & 1);
      float e = 0.0f;
      if (xe && ye) {
        e = E(ax, by) * Fv;
      } else if (!xe && ye) {
        if (x <= w - 3) e = Fv * (E(ax, by) + E(ax + 1, by)) / eps_count(FC(ax, by) + FC(ax + 1, by));
      } else if (xe && !ye) {
        if (y <= h - 3) e = Fv * (E(ax, by) + E(ax, by + 1)) / eps_count(FC(ax, by) + FC(ax, by + 1));
      } else {
        if (x <= w - 3 && y <= h - 3)
          e = Fv * (E(ax, by) + E(ax + 1, by + 1) + E(ax + 1, by) + E(ax, by + 1)) /
              eps_count(FC(ax, by) + FC(ax + 1, by + 1) + FC(ax + 1, by) + FC(ax, by + 1));
      }
      p[i] += e;
    }
  } while (tw.next(a));
}

// the coarse levels of each domain in LDS, one workgroup per domain slot;
// ia: index of p at the domain's first LDS level
template <bool BIG>
__global__ void __launch_bounds__(TPB_C) kb_coarse(StageArgs a, const CoarseArgs *cargs,
                                                   int nslots) {
  const int d = blockIdx.x;
  if (d >= nslots) return;
  const BDom &D = a.dom[d];
  if (!dom_active(D) || D.cfirst >= D.nlev) return;
  const BLev &L = a.lev[d * BMAXL + D.cfirst];
  coarse_vcycle_body<BIG>(cargs[d], L.f, L.p[a.ia[d]]);
}

__device__ __forceinline__ double wsum(double v) {
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  return v;
}

// the domains' solve states from / to one array: a block per domain
static_assert(sizeof(DState) % sizeof(double) == 0, "copied as doubles");
__global__ void __launch_bounds__(64) kb_put_states(DState *const *__restrict__ st,
                                                    const DState *__restrict__ src) {
  double *d = (double *)st[blockIdx.x];
  const double *s = (const double *)&src[blockIdx.x];
  for (unsigned i = threadIdx.x; i < sizeof(DState) / sizeof(double); i += 64) d[i] = s[i];
}
__global__ void __launch_bounds__(64) kb_get_states(DState *const *__restrict__ st,
                                                    DState *__restrict__ dst) {
  const double *s = (const double *)st[blockIdx.x];
  double *d = (double *)&dst[blockIdx.x];
  for (unsigned i = threadIdx.x; i < sizeof(DState) / sizeof(double); i += 64) d[i] = s[i];
}

// The refinement update of refine.hip's k_ir_update for 256 x 8 tiles of
// every domain: ia = e index of level 0; ib bit 0 = x index, bit 1 = add e.
__global__ void __launch_bounds__(B_UPD_W) kb_update(StageArgs a) {
  static_assert(B_UPD_W == kIrCols && B_UPD_H == kIrRows, "blocks of ir_update_column");
  __shared__ double red[B_UPD_W / 64];
  TileWalk tw;
  if (!tw.init(a)) return;
  do {
    const Tile T{tw.d, tw.tx() * B_UPD_W, tw.ty() * B_UPD_H, tw.j};
    const BDom &D = a.dom[T.d];
    if (!dom_active(D)) continue;
    const BLev &L0 = a.lev[T.d * BMAXL];
    const int ie = a.ia[T.d], b = a.ib[T.d];
    const bool ACC = (b >> 1) & 1;
    const double *__restrict__ xa = D.x[b & 1];
    double *__restrict__ xb = D.x[(b & 1) ^ 1];
    const float *__restrict__ e = L0.p[ie];
    float *__restrict__ ez = L0.p[ie ^ 1];
    const float *__restrict__ f = D.rhs;
    const uint8_t *__restrict__ m = L0.mask;
    float *__restrict__ r32 = L0.f;
    const int w = D.w, h = D.h;
    const double ihsq = 1.0 / ((double)L0.hh * (double)L0.hh);
    const int x = T.x0 + threadIdx.x;
    double acc = ACC ? ir_update_column<true>(x, T.y0, xa, xb, e, ez, f, m, r32, w, h, ihsq)
                     : ir_update_column<false>(x, T.y0, xa, xb, e, ez, f, m, r32, w, h, ihsq);
    acc = wsum(acc);
    __syncthreads();
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = acc;
    __syncthreads();
    if (threadIdx.x == 0) {
      double s = 0.0;
      for (int i = 0; i < B_UPD_W / 64; i++) s += red[i];
      D.partial[T.i] = s;
    }
  } while (tw.next(a));
}

// per-domain norm (the order of refine.hip's k_sum_partials) and the
// convergence rule of ubg_mg_ir_solve; ia = 1 for a domain's first update,
// ib = its x index after the update.  One 1024-thread block per domain slot.
__global__ void __launch_bounds__(1024) kb_norm(StageArgs a, int nslots) {
  const int d = blockIdx.x;
  if (d >= nslots) return;
  const BDom &D = a.dom[d];
  if (!dom_active(D)) return;
  const int n = D.gx * D.gy;
  double s = thread_partials(D.partial, n);
  __shared__ double red[16];
  s = wsum(s);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = s;
  __syncthreads();
  if (threadIdx.x != 0) return;
  double n2 = 0.0;
  for (int i = 0; i < 16; i++) n2 += red[i];
  DState &S = *D.st;
  S.xcur = a.ib[d];
  if (a.ia[d]) { // first update: the initial residual
    const double r = sqrt(n2);
    S.r0 = S.ref > 0.0 ? S.ref : r;
    S.iters = 0;
    S.vcycles = 0;
    S.stall = 0;
    S.best = 1.0;
    S.converged = 0;
    if (!isfinite(r)) {
      S.nonfinite = 1;
      S.active = 0;
      return;
    }
    S.rel = r == 0.0 ? 0.0 : r / S.r0;
    if (r == 0.0 || S.rel <= S.tol) { // nothing to do (a warm start may already meet tol)
      S.converged = 1;
      S.active = 0;
    }
    return;
  }
  const double rel = sqrt(n2) / S.r0;
  S.iters += 1;
  S.vcycles += S.k;
  S.rel = rel;
  if (S.iters <= UBG_IR_HISTORY) S.hist[S.iters - 1] = rel;
  if (!isfinite(rel)) {
    S.nonfinite = 1;
    S.active = 0;
    return;
  }
  if (rel <= S.tol) {
    S.converged = 1;
    S.active = 0;
    return;
  }
  if (rel > 0.9 * S.best) {
    if (++S.stall >= 3) S.active = 0;
  } else {
    S.stall = 0;
  }
  S.best = fmin(S.best, rel);
  if (S.iters >= S.max_iter) S.active = 0;
}

// Level-0 copies of up to kCopyJobs domains in one launch (batched
// simulation steps): block (x, j) copies a stride of job j's p (and f when
// its source is set).  The jobs travel as the kernel's argument.
constexpr int kCopyJobs = 64;
struct CopyJob {
  const float *sp, *sf;
  float *dp, *df;
  int n;
};
struct CopyJobs {
  CopyJob j[kCopyJobs];
};
__global__ void __launch_bounds__(256) kb_copy_level0(CopyJobs jobs, int njobs) {
  if ((int)blockIdx.y >= njobs) return;
  const CopyJob &J = jobs.j[blockIdx.y];
  for (int i = blockIdx.x * 256 + threadIdx.x; i < J.n; i += gridDim.x * 256) {
    J.dp[i] = J.sp[i];
    if (J.sf) J.df[i] = J.sf[i];
  }
}

__global__ void __launch_bounds__(256) kb_count(const BDom *dom, int n, int *out,
                                                uint8_t *flags) {
  __shared__ int red[4];
  int c = 0;
  for (int i = threadIdx.x; i < n; i += 256) {
    const int a = dom[i].st->active ? 1 : 0;
    flags[i] = (uint8_t)a;
    c += a;
  }
  for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = c;
  __syncthreads();
  if (threadIdx.x == 0) out[0] = red[0] + red[1] + red[2] + red[3];
}

// the compiled smoother tile shapes
struct Shape {
  int tx, ty;
};
constexpr Shape kShapes[] = {{32, 8}, {64, 4}, {64, 8}, {64, 16}, {128, 4}, {128, 8}, {256, 4}};

void launch_sweep(const Tuning &tn, int blocks, hipStream_t s, const StageArgs &a) {
#define UBG_SW(X, Y)                                                                            \
  if (tn.tx == X && tn.ty == Y) {                                                               \
    hipLaunchKernelGGL((kb_sweep<X, Y>), dim3(blocks), dim3(TPB), 0, s, a);                     \
    return;                                                                                     \
  }
  UBG_SW(32, 8)
  UBG_SW(64, 4)
  UBG_SW(64, 8)
  UBG_SW(64, 16)
  UBG_SW(128, 4)
  UBG_SW(128, 8)
  UBG_SW(256, 4)
#undef UBG_SW
}

bool shape_ok(int tx, int ty) {
  for (const Shape &s : kShapes)
    if (s.tx == tx && s.ty == ty) return true;
  return false;
}

size_t al(size_t n) { return align_up(n, 256); }

// tile shapes of the level passes the tuning may fix (0: chosen per level)
bool pass_rows_ok(int r) { return r == 0 || r == 8 || r == 16 || r == 32; }

} // namespace

// ===========================================================================
// Arena
// ===========================================================================
int Arena::init(size_t bytes) {
  cap_ = al(bytes);
  UBG_HIP(hipMalloc((void **)&base_, cap_));
  free_.clear();
  live_.clear();
  free_[0] = cap_;
  used_ = 0;
  return UBG_OK;
}

void Arena::release() {
  if (base_) (void)hipFree(base_);
  base_ = nullptr;
  free_.clear();
  live_.clear();
  cap_ = used_ = 0;
}

char *Arena::alloc(size_t bytes) {
  bytes = al(bytes ? bytes : 1);
  for (auto it = free_.begin(); it != free_.end(); ++it) {
    if (it->second < bytes) continue;
    size_t off = it->first, sz = it->second;
    free_.erase(it);
    if (sz > bytes) free_[off + bytes] = sz - bytes;
    live_[off] = bytes;
    used_ += bytes;
    return base_ + off;
  }
  return nullptr;
}

void Arena::free(char *p) {
  if (!p) return;
  size_t off = (size_t)(p - base_);
  auto it = live_.find(off);
  if (it == live_.end()) return;
  size_t sz = it->second;
  live_.erase(it);
  used_ -= sz;
  auto nx = free_.lower_bound(off);
  if (nx != free_.end() && off + sz == nx->first) {
    sz += nx->second;
    free_.erase(nx);
  }
  auto pv = free_.lower_bound(off);
  if (pv != free_.begin()) {
    --pv;
    if (pv->first + pv->second == off) {
      pv->second += sz;
      return;
    }
  }
  free_[off] = sz;
}

// ===========================================================================
// shapes, geometries, domains
// ===========================================================================
int batch_shape(int W, int H, BShape *s) {
  if (W < B_MIN_SIZE || H < B_MIN_SIZE)
    return fail(UBG_E_DOMAIN_TOO_SMALL, "batched domains need at least 16 x 16 cells");
  std::vector<int> ws, hs;
  level_sizes(W, H, ws, hs);
  if ((int)ws.size() > BMAXL) return fail(UBG_E_INVALID, "too many levels");
  *s = BShape{};
  s->nlev = (int)ws.size();
  for (int l = 0; l < s->nlev; l++) {
    s->w[l] = ws[l];
    s->h[l] = hs[l];
  }
  // the LDS V-cycle starts where the single-domain solver starts it (the
  // first level of at most kCoarseMaxCells cells: larger LDS levels cost more
  // than their tile passes), or at the first level whose sub-hierarchy fits
  // if that one does not
  s->cfirst = -1;
  int fit = -1;
  size_t fit_bytes = 0;
  for (int l = 1; l <= s->nlev - 2; l++) {
    size_t b = coarse_lds_layout(ws.data(), hs.data(), l, s->nlev, nullptr);
    if (b > LDS_BUDGET) continue;
    if (fit < 0) {
      fit = l;
      fit_bytes = b;
    }
    if ((size_t)ws[l] * hs[l] <= kCoarseMaxCells) {
      s->cfirst = l;
      s->lds_bytes = b;
      break;
    }
  }
  if (s->cfirst < 0 && fit >= 0) {
    s->cfirst = fit;
    s->lds_bytes = fit_bytes;
  }
  if (s->cfirst < 0) return fail(UBG_E_INVALID, "no coarse level fits in LDS");
  for (int l = 0; l < s->nlev; l++) s->geom_bytes += 2 * al((size_t)ws[l] * hs[l]);
  const size_t n0 = (size_t)W * H;
  const int gx = (W + B_UPD_W - 1) / B_UPD_W, gy = (H + B_UPD_H - 1) / B_UPD_H;
  size_t b = 2 * al(n0 * 8) + al(n0 * 4) + al((size_t)gx * gy * 8) + al(sizeof(DState));
  for (int l = 0; l <= s->cfirst; l++) b += 3 * al((size_t)ws[l] * hs[l] * 4);
  s->dom_bytes = b;
  return UBG_OK;
}

Staging::~Staging() {
  for (Block &b : blocks_) {
    (void)hipHostFree(b.host);
    (void)hipFree(b.dev);
  }
}

int Staging::reserve(size_t bytes) {
  if (!blocks_.empty() && blocks_.back().cap - blocks_.back().used >= bytes) return UBG_OK;
  Block b;
  for (const Block &q : blocks_) b.cap += q.cap;
  b.cap = std::max(b.cap, al(bytes));
  UBG_HIP(hipHostMalloc((void **)&b.host, b.cap, hipHostMallocDefault));
  const hipError_t e = hipMalloc((void **)&b.dev, b.cap);
  if (e != hipSuccess) {
    (void)hipHostFree(b.host);
    UBG_HIP(e);
  }
  blocks_.push_back(b);
  return UBG_OK;
}

int Staging::carve(size_t bytes, char **host, char **dev) {
  bytes = al(bytes);
  UBG_TRY(reserve(bytes));
  Block &b = blocks_.back();
  *host = b.host + b.used;
  *dev = b.dev + b.used;
  b.used += bytes;
  return UBG_OK;
}

UploadRing::~UploadRing() {
  for (Slot &q : slot_)
    if (q.used) (void)hipEventDestroy(q.used);
}

int UploadRing::reserve(Staging &st, size_t bytes) {
  for (Slot &q : slot_) {
    UBG_HIP(hipEventCreateWithFlags(&q.used, hipEventDisableTiming));
    UBG_TRY(st.carve(bytes, &q.host, &q.dev));
    q.cap = al(bytes);
  }
  return UBG_OK;
}

int UploadRing::put(Staging &st, const void *data, size_t bytes, hipStream_t s, char **dev) {
  if (cur_ >= 0) UBG_HIP(hipEventRecord(slot_[cur_].used, s));
  cur_ = (cur_ + 1) % SLOTS;
  Slot &q = slot_[cur_];
  UBG_HIP(hipEventSynchronize(q.used)); // at once unless recorded and not passed
  if (bytes > q.cap) {
    const size_t cap = 2 * bytes;
    UBG_TRY(st.carve(cap, &q.host, &q.dev));
    q.cap = al(cap);
  }
  *dev = q.dev;
  if (!bytes) return UBG_OK;
  std::memcpy(q.host, data, bytes);
  UBG_HIP(hipMemcpyAsync(q.dev, q.host, bytes, hipMemcpyHostToDevice, s));
  return UBG_OK;
}

// sizes of the uploads for n member domains
static size_t tables_bytes(size_t n) {
  return al(n * BMAXL * sizeof(BLev)) + al(n * sizeof(BDom)) + n * sizeof(CoarseArgs);
}
static size_t states_bytes(size_t n) { return al(n * sizeof(DState *)) + n * sizeof(DState); }

BatchEngine::~BatchEngine() { drop_graphs(); }

int BatchEngine::init(hipStream_t s, const ubg_params &prm, int vcycles_per_step, int members) {
  stream_ = s;
  prm_ = prm;
  k_ = vcycles_per_step;
  // tile maps: sweep, residual and prolongation stages, the two passes of a
  // level, the update; index rows: two steps of domains of eight levels, to 1 MB
  const size_t n = (size_t)members, maps = (tiled() ? 5 : 3) * BMAXL + 1;
  const size_t stages = tiled() ? 2 * 8 + 1 : 8 * ((size_t)prm_.nu_pre + prm_.nu_post + 2) + 1;
  const size_t tab = tables_bytes(n), off = maps * (3 * n + 1) * sizeof(int),
               idx = std::min(2 * (k_ * stages + 2) * 2 * n, size_t(1) << 20),
               st = states_bytes(n);
  UBG_TRY(staging_.reserve(UploadRing::SLOTS * (al(tab) + al(off) + al(idx) + al(st)) + al(n) +
                           al(sizeof(int))));
  UBG_TRY(tab_ring_.reserve(staging_, tab));
  UBG_TRY(off_ring_.reserve(staging_, off));
  UBG_TRY(idx_ring_.reserve(staging_, idx));
  UBG_TRY(st_ring_.reserve(staging_, st));
  UBG_TRY(reserve_active(n));
  char *host, *dev;
  UBG_TRY(staging_.carve(sizeof(int), &host, &dev));
  count_host_ = (int *)host;
  d_count_ = (int *)dev;
  *count_host_ = 0;
  static const bool attr_set = [] { // more than 64 KiB of LDS
    for (auto k : {kb_coarse<false>, kb_coarse<true>})
      (void)hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                (int)LDS_BUDGET);
    return true;
  }();
  (void)attr_set;
  return UBG_OK;
}

int BatchEngine::geom_create(Arena &arena, int W, int H, const float *flag, BGeom **out,
                             bool need_ring) {
  BShape sh;
  UBG_TRY(batch_shape(W, H, &sh));
  std::vector<uint8_t> f8;
  UBG_TRY(validate_flag(flag, (size_t)W * H, f8));
  bool ring = true;
  for (int x = 0; x < W; x++)
    if (!f8[x] || !f8[(size_t)(H - 1) * W + x]) ring = false;
  for (int y = 0; y < H; y++)
    if (!f8[(size_t)y * W] || !f8[(size_t)y * W + W - 1]) ring = false;
  if (need_ring && !ring)
    return fail(UBG_E_FLAG_VALUE, "the outer ring of a solve domain must be fluid");
  auto *g = new BGeom();
  g->ring_fluid = ring;
  g->W = W;
  g->H = H;
  g->nlev = sh.nlev;
  g->cfirst = sh.cfirst;
  g->lds_bytes = sh.lds_bytes;
  g->bytes = sh.geom_bytes;
  g->mem = arena.alloc(g->bytes);
  if (!g->mem) {
    delete g;
    return fail(UBG_E_BUDGET, "device arena full (geometry)");
  }
  char *q = g->mem;
  for (int l = 0; l < g->nlev; l++) {
    g->w[l] = sh.w[l];
    g->h[l] = sh.h[l];
    size_t n = (size_t)g->w[l] * g->h[l];
    g->flag[l] = (uint8_t *)q;
    q += al(n);
    g->mask[l] = (uint8_t *)q;
    q += al(n);
  }
  UBG_HIP(hipMemcpyAsync(g->flag[0], f8.data(), f8.size(), hipMemcpyHostToDevice, stream_));
  std::vector<Level> lv((size_t)g->nlev);
  for (int l = 0; l < g->nlev; l++) {
    lv[l].w = g->w[l];
    lv[l].h = g->h[l];
    lv[l].flag = g->flag[l];
    lv[l].mask = g->mask[l];
  }
  launch_classify(lv.data(), g->nlev, nullptr, false, stream_);
  UBG_TRY(check_launch());
  UBG_HIP(hipStreamSynchronize(stream_)); // f8 is a host temporary
  g->refs = 1;
  *out = g;
  return UBG_OK;
}

void BatchEngine::geom_release(Arena &arena, BGeom *g) {
  if (!g || --g->refs > 0) return;
  arena.free(g->mem);
  delete g;
}

int BatchEngine::domain_create(Arena &arena, BGeom *g, float h, BDomain **out, hipStream_t s) {
  BShape sh;
  UBG_TRY(batch_shape(g->W, g->H, &sh));
  auto *d = new BDomain();
  d->id = next_id_++;
  d->g = g;
  d->h = h;
  d->bytes = sh.dom_bytes;
  d->mem = arena.alloc(d->bytes);
  if (!d->mem) {
    delete d;
    return fail(UBG_E_BUDGET, "device arena full (domain)");
  }
  const size_t n0 = (size_t)g->W * g->H;
  d->gx = (g->W + B_UPD_W - 1) / B_UPD_W;
  d->gy = (g->H + B_UPD_H - 1) / B_UPD_H;
  char *q = d->mem;
  d->x[0] = (double *)q;
  q += al(n0 * 8);
  d->x[1] = (double *)q;
  q += al(n0 * 8);
  d->rhs = (float *)q;
  q += al(n0 * 4);
  d->partial = (double *)q;
  q += al((size_t)d->gx * d->gy * 8);
  d->st = (DState *)q;
  q += al(sizeof(DState));
  for (int l = 0; l <= g->cfirst; l++) {
    size_t n = (size_t)g->w[l] * g->h[l];
    d->p[l][0] = (float *)q;
    q += al(n * 4);
    d->p[l][1] = (float *)q;
    q += al(n * 4);
    d->f[l] = (float *)q;
    q += al(n * 4);
  }
  // h of each level: h_c = h * (W_l - 1) / (W_{l+1} - 1) (pressure_solver.cpp:229)
  d->hh[0] = h;
  for (int l = 1; l < g->nlev; l++) d->hh[l] = d->hh[l - 1] * (g->w[l - 1] - 1.0f) / (g->w[l] - 1.0f);
  UBG_HIP(hipMemsetAsync(d->mem, 0, d->bytes, s ? s : stream_));
  g->refs++;
  *out = d;
  return UBG_OK;
}

void BatchEngine::domain_release(Arena &arena, BDomain *d) {
  if (!d) return;
  arena.free(d->mem);
  geom_release(arena, d->g);
  delete d;
}

int BatchEngine::domain_set_rhs(BDomain *d, const float *rhs) {
  const size_t n = (size_t)d->g->W * d->g->H;
  for (size_t i = 0; i < n; i++)
    if (!std::isfinite(rhs[i])) return fail(UBG_E_NONFINITE, "rhs has a non-finite value");
  UBG_HIP(hipMemcpyAsync(d->rhs, rhs, n * 4, hipMemcpyHostToDevice, stream_));
  UBG_HIP(hipStreamSynchronize(stream_));
  return UBG_OK;
}

int BatchEngine::domain_set_guess(BDomain *d, const double *x) {
  const size_t n = (size_t)d->g->W * d->g->H;
  if (x) {
    for (size_t i = 0; i < n; i++)
      if (!std::isfinite(x[i])) return fail(UBG_E_NONFINITE, "guess has a non-finite value");
    UBG_HIP(hipMemcpyAsync(d->x[d->xcur], x, n * 8, hipMemcpyHostToDevice, stream_));
  } else {
    launch_fill_f64(d->x[d->xcur], n, 0.0, stream_);
    UBG_TRY(check_launch());
  }
  UBG_HIP(hipStreamSynchronize(stream_));
  return UBG_OK;
}

// a domain's solve state before its first update
static DState start_state(double tol, int max_iter, double ref, int k, int xcur) {
  DState st{};
  st.active = 1;
  st.tol = tol;
  st.ref = ref;
  st.max_iter = max_iter;
  st.k = k;
  st.best = 1.0;
  st.rel = 1.0;
  st.xcur = xcur;
  return st;
}

int BatchEngine::domain_start(BDomain *d, double tol, int max_iter, double ref, hipStream_t s) {
  if (!s) s = stream_;
  const DState st = start_state(tol, max_iter, ref, k_, d->xcur);
  UBG_HIP(hipMemcpyAsync(d->st, &st, sizeof(st), hipMemcpyHostToDevice, s));
  UBG_HIP(hipStreamSynchronize(s));
  return UBG_OK;
}

int BatchEngine::domain_read_state(BDomain *d, DState *out, hipStream_t s) {
  if (!s) s = stream_;
  UBG_HIP(hipMemcpyAsync(out, d->st, sizeof(DState), hipMemcpyDeviceToHost, s));
  UBG_HIP(hipStreamSynchronize(s));
  return UBG_OK;
}

int BatchEngine::start_all(const std::vector<BDomain *> &doms, double tol, int max_iter) {
  const size_t n = doms.size(), ptr_bytes = al(n * sizeof(DState *));
  if (!n) return UBG_OK;
  if (n == 1) return domain_start(doms[0], tol, max_iter); // one copy instead of a table and a launch
  std::vector<char> blob(states_bytes(n));
  for (size_t i = 0; i < n; i++) {
    ((DState **)blob.data())[i] = doms[i]->st;
    DState &st = ((DState *)(blob.data() + ptr_bytes))[i];
    st = start_state(tol, max_iter, 0.0, k_, doms[i]->xcur);
  }
  char *dev = nullptr;
  UBG_TRY(st_ring_.put(staging_, blob.data(), blob.size(), stream_, &dev));
  hipLaunchKernelGGL(kb_put_states, dim3((unsigned)n), dim3(64), 0, stream_, (DState *const *)dev,
                     (const DState *)(dev + ptr_bytes));
  return check_launch();
}

int BatchEngine::read_states(const std::vector<BDomain *> &doms, std::vector<DState> &out) {
  const size_t n = doms.size(), ptr_bytes = al(n * sizeof(DState *));
  out.resize(n);
  if (!n) return UBG_OK;
  if (n == 1) return domain_read_state(doms[0], out.data());
  std::vector<char> blob(states_bytes(n));
  for (size_t i = 0; i < n; i++) ((DState **)blob.data())[i] = doms[i]->st;
  char *dev = nullptr;
  UBG_TRY(st_ring_.put(staging_, blob.data(), blob.size(), stream_, &dev));
  hipLaunchKernelGGL(kb_get_states, dim3((unsigned)n), dim3(64), 0, stream_, (DState *const *)dev,
                     (DState *)(dev + ptr_bytes));
  UBG_TRY(check_launch());
  UBG_HIP(hipMemcpyAsync(out.data(), dev + ptr_bytes, n * sizeof(DState), hipMemcpyDeviceToHost,
                         stream_));
  UBG_HIP(hipStreamSynchronize(stream_));
  return UBG_OK;
}

int BatchEngine::domain_get_solution(BDomain *d, double *x, hipStream_t s) {
  if (!s) s = stream_;
  const size_t n = (size_t)d->g->W * d->g->H;
  UBG_HIP(hipMemcpyAsync(x, d->x[d->xcur], n * 8, hipMemcpyDeviceToHost, s));
  UBG_HIP(hipStreamSynchronize(s));
  return UBG_OK;
}

int BatchEngine::domain_set_level0(BDomain *d, const float *p, const float *f,
                                   hipMemcpyKind kind, hipStream_t s) {
  if (!s) s = stream_;
  const size_t n = (size_t)d->g->W * d->g->H;
  float *p0 = d->p[0][d->cur[0]];
  if (p) UBG_HIP(hipMemcpyAsync(p0, p, n * 4, kind, s));
  else launch_fill_f32(p0, n, 0.0f, s);
  if (f) UBG_HIP(hipMemcpyAsync(d->f[0], f, n * 4, kind, s));
  UBG_TRY(check_launch());
  if (kind != hipMemcpyDeviceToDevice) UBG_HIP(hipStreamSynchronize(s));
  return UBG_OK;
}

int BatchEngine::domain_get_pressure(BDomain *d, float *p, hipMemcpyKind kind, hipStream_t s) {
  if (!s) s = stream_;
  const size_t n = (size_t)d->g->W * d->g->H;
  UBG_HIP(hipMemcpyAsync(p, d->p[0][d->cur[0]], n * 4, kind, s));
  if (kind != hipMemcpyDeviceToDevice) UBG_HIP(hipStreamSynchronize(s));
  return UBG_OK;
}

// ===========================================================================
// member tables, tiles, schedules
// ===========================================================================
void BatchEngine::drop_graphs() {
  for (auto &kv : graphs_) {
    if (kv.second.exec) (void)hipGraphExecDestroy(kv.second.exec);
    if (kv.second.d_idx) (void)hipFree(kv.second.d_idx);
  }
  graphs_.clear();
}

int BatchEngine::set_members(const std::vector<BDomain *> &running,
                             const std::vector<BDomain *> &fresh) {
  // by their ids: a released member's address may be another domain's by now
  std::vector<uint64_t> ids;
  for (const auto *v : {&running, &fresh})
    for (const BDomain *d : *v) ids.push_back(d->id);
  if (ids == ids_ && running.size() == run_.size() && d_lev_) return UBG_OK;
  run_ = running;
  fresh_ = fresh;
  all_ = running;
  all_.insert(all_.end(), fresh.begin(), fresh.end());
  ids_ = std::move(ids);
  drop_graphs();
  int rc = build_tables();
  if (rc == UBG_OK) rc = build_tiles();
  if (rc != UBG_OK) invalidate_members(); // the tables are an earlier set's
  return rc;
}

int BatchEngine::reserve_active(size_t n) {
  char *host, *dev;
  UBG_TRY(staging_.carve(n, &host, &dev));
  h_active_ = (uint8_t *)host;
  d_active_ = (uint8_t *)dev;
  std::memset(h_active_, 0, n);
  act_cap_ = n;
  return UBG_OK;
}

int BatchEngine::build_tables() {
  const size_t n = all_.size();
  if (n > act_cap_) UBG_TRY(reserve_active(2 * n));
  const size_t lev_bytes = al(n * BMAXL * sizeof(BLev)), dom_bytes = al(n * sizeof(BDom));
  std::vector<char> blob(tables_bytes(n));
  BLev *lev = (BLev *)blob.data();
  BDom *dom = (BDom *)(blob.data() + lev_bytes);
  CoarseArgs *ca = (CoarseArgs *)(blob.data() + lev_bytes + dom_bytes);
  coarse_lds_ = 0;
  coarse_big_ = false;
  lmax_ = 0;
  for (size_t s = 0; s < n; s++) {
    const BDomain &D = *all_[s];
    const BGeom &G = *D.g;
    for (int l = 0; l < G.nlev; l++) {
      BLev &L = lev[s * BMAXL + l];
      L.p[0] = l <= G.cfirst ? D.p[l][0] : nullptr;
      L.p[1] = l <= G.cfirst ? D.p[l][1] : nullptr;
      L.f = l <= G.cfirst ? D.f[l] : nullptr;
      L.mask = G.mask[l];
      L.w = G.w[l];
      L.h = G.h[l];
      L.hh = D.hh[l];
      L.ihsq = 1.0f / D.hh[l] / D.hh[l];
    }
    BDom &B = dom[s];
    B.st = D.st;
    B.x[0] = D.x[0];
    B.x[1] = D.x[1];
    B.rhs = D.rhs;
    B.partial = D.partial;
    B.w = G.W;
    B.h = G.H;
    B.gx = D.gx;
    B.gy = D.gy;
    B.nlev = G.nlev;
    B.cfirst = G.cfirst;
    CoarseArgs &a = ca[s];
    a = CoarseArgs{};
    coarse_lds_layout(G.w, G.h, G.cfirst, G.nlev, &a);
    a.n = G.nlev - 1 - G.cfirst;
    for (int k = 0; k < a.n; k++) {
      const int l = G.cfirst + k;
      a.w[k] = G.w[l];
      a.h[k] = G.h[l];
      a.mask[k] = G.mask[l];
      a.hh[k] = D.hh[l];
      a.ihsq[k] = 1.0f / D.hh[l] / D.hh[l];
    }
    a.nu_pre = prm_.nu_pre;
    a.nu_post = prm_.nu_post;
    a.nu_coarse = prm_.nu_coarse;
    a.alpha = prm_.alpha;
    if (s < run_.size()) {
      coarse_lds_ = std::max(coarse_lds_, G.lds_bytes);
      coarse_big_ = coarse_big_ || coarse_big(G.w[G.cfirst], G.h[G.cfirst]);
      lmax_ = std::max(lmax_, G.cfirst);
    }
  }
  if (n) {
    char *dev = nullptr;
    UBG_TRY(tab_ring_.put(staging_, blob.data(), blob.size(), stream_, &dev));
    d_lev_ = (BLev *)dev;
    d_dom_ = (BDom *)(dev + lev_bytes);
    d_cargs_ = (CoarseArgs *)(dev + lev_bytes + dom_bytes);
  }
  return UBG_OK;
}

// Per stage kind and level: the prefix of tile counts over the member slots
// and each domain's tiles per row; kernels locate their tile from these, so
// a member change rebuilds O(domains x levels) integers, not tile lists.
int BatchEngine::build_tiles() {
  h_off_.clear();
  // per span: tile prefix over the domain slots [nd + 1], tiles per row [nd]
  // and the tile width [nd] (fused passes; 0 elsewhere)
  auto span = [&](Span &sp, int nd, auto tiles_of) {
    sp.off = h_off_.size();
    sp.nd = nd;
    h_off_.resize(sp.off + 3 * (size_t)nd + 1);
    int *pre = h_off_.data() + sp.off, *ntx = pre + nd + 1, *otx = ntx + nd;
    long tot = 0;
    for (int s = 0; s < nd; s++) {
      int nx = 0, ny = 0, ox = 0;
      tiles_of(s, nx, ny, ox);
      pre[s] = (int)tot;
      ntx[s] = nx > 0 ? nx : 1;
      otx[s] = ox;
      tot += (long)nx * ny;
    }
    pre[nd] = (int)tot;
    sp.n = (int)tot;
  };
  auto cdiv = [](int a, int b) { return a > 0 ? (a + b - 1) / b : 0; };
  const int tx = tune_.tx, ty = tune_.ty;
  const int nr = (int)run_.size();
  for (int l = 0; l < BMAXL; l++) {
    span(sw_[l], nr, [&](int s, int &nx, int &ny, int &) {
      const BGeom &G = *run_[s]->g;
      if (l >= G.cfirst) return;
      nx = cdiv(G.w[l], tx);
      ny = cdiv(G.h[l], ty);
    });
    span(rr_[l], nr, [&](int s, int &nx, int &ny, int &) {
      const BGeom &G = *run_[s]->g;
      if (l >= G.cfirst) return;
      nx = cdiv(G.w[l + 1] - 2, RCX);
      ny = cdiv(G.h[l + 1] - 2, RCY);
    });
    span(pc_[l], nr, [&](int s, int &nx, int &ny, int &) {
      const BGeom &G = *run_[s]->g;
      if (l >= G.cfirst) return;
      nx = cdiv(G.w[l] - 2, PCW);
      ny = cdiv(G.h[l] - 2, PCH);
    });
  }
  // Level passes: one tile shape per pass of a level, by the tuning or by the
  // members' tiles together; each domain's columns split evenly.
  auto passes = [&](Span *out, bool pre, int nu) {
    for (int l = 0; l < BMAXL && tiled(); l++) {
      auto tiles = [&](PassShape shape) {
        int ox = 0, oy = 0;
        pass_tile(shape, pre, nu, &ox, &oy);
        long t = 0;
        for (int s = 0; s < nr; s++) {
          const BGeom &G = *run_[s]->g;
          if (l < G.cfirst) t += (long)cdiv(G.w[l], ox) * cdiv(G.h[l], oy);
        }
        return t;
      };
      PassShape shape = pass_shape(tiles(PASS_TINY), tiles(PASS_SMALL));
      if (tune_.prow) shape = tune_.prow == 8 ? PASS_SMALL : (tune_.prow == 16 ? PASS_MID : PASS_BIG);
      int otx = 0, oty = 0;
      pass_tile(shape, pre, nu, &otx, &oty);
      out[l].oty = oty;
      out[l].shape = shape;
      span(out[l], nr, [&](int s, int &nx, int &ny, int &ox) {
        const BGeom &G = *run_[s]->g;
        if (l >= G.cfirst) return;
        nx = cdiv(G.w[l], otx);
        ox = (cdiv(G.w[l], nx) + 1) & ~1;
        nx = cdiv(G.w[l], ox);
        ny = cdiv(G.h[l], oty);
      });
    }
  };
  passes(tp_, true, prm_.nu_pre);
  passes(tq_, false, prm_.nu_post);
  span(upd_, (int)all_.size(), [&](int s, int &nx, int &ny, int &) {
    nx = all_[s]->gx;
    ny = all_[s]->gy;
  });
  return off_ring_.put(staging_, h_off_.data(), h_off_.size() * sizeof(int), stream_, (char **)&d_off_);
}

enum { ST_SWEEP, ST_RR, ST_PC, ST_COARSE, ST_UPDATE, ST_NORM, ST_TPRE, ST_TPOST };

// One V-cycle of the running members in the tiled mode (the per-level
// passes of solveLevel, pressure_solver.cpp:201-248), simulated on (and
// advancing) the domains' host index state.
void BatchEngine::gen_vcycle_tiled(std::vector<StageRec> &st, std::vector<uint8_t> &idx) {
  const size_t n = all_.size();
  const size_t nr = run_.size();
  auto row = [&](int kind, int level) -> std::pair<uint8_t *, uint8_t *> {
    size_t off = idx.size();
    idx.resize(off + 2 * n, 0);
    st.push_back(StageRec{kind, level, off});
    return {idx.data() + off, idx.data() + off + n};
  };
  // per level one pass on the way down and one on the way up, each flipping
  // the level's p
  auto pass_row = [&](int kind, int l) {
    auto r = row(kind, l);
    for (size_t d = 0; d < nr; d++)
      if (l < run_[d]->g->cfirst) {
        r.first[d] = (uint8_t)run_[d]->cur[l];
        r.second[d] = (uint8_t)run_[d]->cur[l + 1];
        run_[d]->cur[l] ^= 1;
      }
  };
  for (int l = 0; l < lmax_; l++)
    if (tp_[l].n) pass_row(ST_TPRE, l);
  {
    auto r = row(ST_COARSE, 0);
    for (size_t d = 0; d < nr; d++) r.first[d] = (uint8_t)run_[d]->cur[run_[d]->g->cfirst];
  }
  for (int l = lmax_ - 1; l >= 0; l--)
    if (tq_[l].n) pass_row(ST_TPOST, l);
}

// The stage sequence of nsteps refinement steps and, per stage, the two
// per-domain index rows, simulated from (and advancing) the domains' host
// index state: a sweep reads p[cur] and writes p[cur^1]; the update reads
// e = p0[cur] and x[xcur], zeroes p0[cur^1], writes x[xcur^1].
void BatchEngine::gen_steps(int nsteps, std::vector<StageRec> &st, std::vector<uint8_t> &idx,
                            bool all_fresh) {
  const size_t n = all_.size();
  const size_t nr = all_fresh ? 0 : run_.size();
  auto row = [&](int kind, int level) -> std::pair<uint8_t *, uint8_t *> {
    size_t off = idx.size();
    idx.resize(off + 2 * n, 0);
    st.push_back(StageRec{kind, level, off});
    return {idx.data() + off, idx.data() + off + n};
  };
  for (int step = 0; step < nsteps; step++) {
    const bool with_fresh = step == 0 && (all_fresh || !fresh_.empty());
    for (int v = 0; v < k_ && nr && tiled(); v++) gen_vcycle_tiled(st, idx);
    for (int v = 0; v < k_ && nr && !tiled(); v++) {
      for (int l = 0; l < lmax_; l++) {
        if (!sw_[l].n && !rr_[l].n) continue;
        for (int s = 0; s < prm_.nu_pre; s++) {
          auto r = row(ST_SWEEP, l);
          for (size_t d = 0; d < nr; d++)
            if (l < run_[d]->g->cfirst) {
              r.first[d] = (uint8_t)run_[d]->cur[l];
              run_[d]->cur[l] ^= 1;
            }
        }
        auto r = row(ST_RR, l);
        for (size_t d = 0; d < nr; d++)
          if (l < run_[d]->g->cfirst) {
            r.first[d] = (uint8_t)run_[d]->cur[l];
            r.second[d] = (uint8_t)run_[d]->cur[l + 1];
          }
      }
      {
        auto r = row(ST_COARSE, 0);
        for (size_t d = 0; d < nr; d++) r.first[d] = (uint8_t)run_[d]->cur[run_[d]->g->cfirst];
      }
      for (int l = lmax_ - 1; l >= 0; l--) {
        if (!pc_[l].n && !sw_[l].n) continue;
        auto r = row(ST_PC, l);
        for (size_t d = 0; d < nr; d++)
          if (l < run_[d]->g->cfirst) {
            r.first[d] = (uint8_t)run_[d]->cur[l];
            r.second[d] = (uint8_t)run_[d]->cur[l + 1];
          }
        for (int s = 0; s < prm_.nu_post; s++) {
          auto q = row(ST_SWEEP, l);
          for (size_t d = 0; d < nr; d++)
            if (l < run_[d]->g->cfirst) {
              q.first[d] = (uint8_t)run_[d]->cur[l];
              run_[d]->cur[l] ^= 1;
            }
        }
      }
    }
    auto u = row(ST_UPDATE, 0);
    for (size_t d = 0; d < all_.size(); d++) {
      BDomain &D = *all_[d];
      const bool fresh = with_fresh && d >= nr;
      if (!fresh && d >= nr) continue; // fresh members join later steps only as running
      u.first[d] = (uint8_t)D.cur[0];
      u.second[d] = (uint8_t)(D.xcur | (fresh ? 0 : 2));
    }
    auto m = row(ST_NORM, 0);
    for (size_t d = 0; d < all_.size(); d++) {
      BDomain &D = *all_[d];
      const bool fresh = with_fresh && d >= nr;
      if (!fresh && d >= nr) continue;
      D.cur[0] ^= 1;
      D.xcur ^= 1;
      m.first[d] = fresh ? 1 : 0;
      m.second[d] = (uint8_t)D.xcur;
    }
  }
}

int BatchEngine::launch_stages(const std::vector<StageRec> &st, const uint8_t *d_idx) {
  const int n = (int)all_.size();
  auto grid = [&](int ntiles) {
    int b = tune_.blocks > 0 ? std::min(ntiles, tune_.blocks) : ntiles;
    return std::max(b, 1);
  };
  auto use = [&](StageArgs &a, const Span &sp) {
    a.off = d_off_ + sp.off;
    a.ndom = sp.nd;
    a.ntiles = sp.n;
  };
  for (const StageRec &r : st) {
    StageArgs a{};
    a.lev = d_lev_;
    a.dom = d_dom_;
    a.level = r.level;
    a.ia = d_idx + r.off;
    a.ib = d_idx + r.off + n;
    a.alpha = prm_.alpha;
    switch (r.kind) {
    case ST_SWEEP:
      use(a, sw_[r.level]);
      if (a.ntiles) launch_sweep(tune_, grid(a.ntiles), stream_, a);
      break;
    case ST_RR:
      use(a, rr_[r.level]);
      if (a.ntiles) hipLaunchKernelGGL(kb_rr, dim3(grid(a.ntiles)), dim3(TPB), 0, stream_, a);
      break;
    case ST_PC:
      use(a, pc_[r.level]);
      if (a.ntiles) hipLaunchKernelGGL(kb_pc, dim3(grid(a.ntiles)), dim3(TPB), 0, stream_, a);
      break;
    case ST_TPRE:
    case ST_TPOST: {
      const bool pre = r.kind == ST_TPRE;
      const Span &sp = pre ? tp_[r.level] : tq_[r.level];
      use(a, sp);
      a.oty = sp.oty;
      if (a.ntiles)
        launch_batch_pass(sp.shape, pre, pre ? prm_.nu_pre : prm_.nu_post, zg0_, grid(a.ntiles),
                          stream_, a);
      break;
    }
    case ST_COARSE:
      if (!run_.empty())
        hipLaunchKernelGGL((coarse_big_ ? kb_coarse<true> : kb_coarse<false>),
                           dim3((unsigned)run_.size()), dim3(TPB_C), coarse_lds_, stream_, a,
                           (const CoarseArgs *)d_cargs_, (int)run_.size());
      break;
    case ST_UPDATE:
      use(a, upd_);
      if (a.ntiles) hipLaunchKernelGGL(kb_update, dim3(grid(a.ntiles)), dim3(B_UPD_W), 0, stream_, a);
      break;
    case ST_NORM:
      hipLaunchKernelGGL(kb_norm, dim3(n), dim3(1024), 0, stream_, a, n);
      break;
    }
  }
  hipLaunchKernelGGL(kb_count, dim3(1), dim3(256), 0, stream_, (const BDom *)d_dom_, n, d_count_,
                     d_active_);
  UBG_TRY(check_launch());
  UBG_HIP(hipMemcpyAsync(count_host_, d_count_, sizeof(int), hipMemcpyDeviceToHost, stream_));
  UBG_HIP(hipMemcpyAsync(h_active_, d_active_, (size_t)n, hipMemcpyDeviceToHost, stream_));
  return UBG_OK;
}

int BatchEngine::upload_idx(const std::vector<uint8_t> &idx, uint8_t **d_idx) {
  return idx_ring_.put(staging_, idx.data(), idx.size(), stream_, (char **)d_idx);
}

int BatchEngine::enqueue_steps(int nsteps) {
  if (all_.empty()) {
    *count_host_ = 0;
    return UBG_OK;
  }
  if (!fresh_.empty() && nsteps != 1)
    return fail(UBG_E_STATE, "members with a pending first update take one step at a time");
  std::vector<StageRec> st;
  std::vector<uint8_t> idx;
  gen_steps(nsteps, st, idx);
  uint8_t *d_idx = nullptr;
  UBG_TRY(upload_idx(idx, &d_idx));
  UBG_TRY(launch_stages(st, d_idx));
  return UBG_OK;
}

int BatchEngine::enqueue_first_update() {
  if (all_.empty()) {
    *count_host_ = 0;
    return UBG_OK;
  }
  std::vector<StageRec> st;
  std::vector<uint8_t> idx;
  gen_steps(1, st, idx, true);
  uint8_t *d_idx = nullptr;
  UBG_TRY(upload_idx(idx, &d_idx));
  UBG_TRY(launch_stages(st, d_idx));
  return UBG_OK;
}

std::string BatchEngine::state_key() const {
  std::string k;
  k.reserve(all_.size() * (BMAXL + 1));
  for (const BDomain *d : all_) {
    for (int l = 0; l < BMAXL; l++) k.push_back((char)('0' + d->cur[l]));
    k.push_back((char)('0' + d->xcur));
  }
  return k;
}

// The stages that `gen` makes, as a captured graph per index state and `what`
// (their index rows in a device buffer of the graph's own), replayed
template <class Gen> int BatchEngine::replay(const std::string &what, Gen gen) {
  const std::string key = state_key() + what;
  std::vector<std::array<int, BMAXL + 1>> start;
  for (BDomain *d : all_) {
    std::array<int, BMAXL + 1> c;
    std::copy(d->cur, d->cur + BMAXL, c.begin());
    c[BMAXL] = d->xcur;
    start.push_back(c);
  }
  // the host index state moves on as the schedule does, unless it cannot run
  std::vector<StageRec> st;
  std::vector<uint8_t> idx;
  gen(st, idx);
  auto undo = [&] {
    for (size_t i = 0; i < all_.size(); i++) {
      std::copy(start[i].begin(), start[i].end() - 1, all_[i]->cur);
      all_[i]->xcur = start[i][BMAXL];
    }
  };
  auto it = graphs_.find(key);
  if (it == graphs_.end()) {
    Graph g;
    const int rc = capture(st, idx, &g);
    if (rc != UBG_OK) {
      undo();
      return rc;
    }
    it = graphs_.emplace(key, g).first;
  }
  const hipError_t e = hipGraphLaunch(it->second.exec, stream_);
  if (e != hipSuccess) undo();
  UBG_HIP(e);
  return UBG_OK;
}

int BatchEngine::capture(const std::vector<StageRec> &st, const std::vector<uint8_t> &idx,
                         Graph *g) {
  UBG_HIP(hipMalloc((void **)&g->d_idx, std::max<size_t>(idx.size(), 1)));
  hipError_t e = hipMemcpy(g->d_idx, idx.data(), idx.size(), hipMemcpyHostToDevice);
  hipGraph_t graph = nullptr;
  int rc = UBG_OK;
  if (e == hipSuccess) e = hipStreamBeginCapture(stream_, hipStreamCaptureModeThreadLocal);
  if (e == hipSuccess) {
    rc = launch_stages(st, g->d_idx);
    e = hipStreamEndCapture(stream_, &graph);
  }
  if (rc == UBG_OK && e == hipSuccess) e = hipGraphInstantiate(&g->exec, graph, nullptr, nullptr, 0);
  if (graph) (void)hipGraphDestroy(graph);
  if (rc == UBG_OK && e == hipSuccess) return UBG_OK;
  (void)hipFree(g->d_idx);
  return rc != UBG_OK ? rc : fail(UBG_E_HIP, std::string("graph capture: ") + hipGetErrorString(e));
}

int BatchEngine::replay_steps(int nsteps) {
  if (!fresh_.empty()) return fail(UBG_E_STATE, "graph replay needs every member running");
  return replay("/" + std::to_string(nsteps),
                [&](std::vector<StageRec> &st, std::vector<uint8_t> &idx) { gen_steps(nsteps, st, idx); });
}

int BatchEngine::enqueue_vcycles(int ncycles, bool zg) {
  if (!tiled() || prm_.nu_pre < 1 || prm_.nu_post < 1)
    return fail(UBG_E_INVALID, "projection batches need 1..3 pre- and post-smoothing sweeps");
  if (!fresh_.empty()) return fail(UBG_E_STATE, "projection batches take running members only");
  if (run_.empty() || ncycles <= 0) return UBG_OK;
  zg0_ = zg;
  const int rc = replay("/v" + std::to_string(ncycles) + (zg ? "z" : "n"),
                        [&](std::vector<StageRec> &st, std::vector<uint8_t> &idx) {
                          for (int v = 0; v < ncycles; v++) gen_vcycle_tiled(st, idx);
                        });
  zg0_ = false;
  return rc;
}

std::vector<BDomain *> BatchEngine::active_members() const {
  std::vector<BDomain *> out;
  for (size_t i = 0; i < all_.size(); i++)
    if (h_active_ && h_active_[i]) out.push_back(all_[i]);
  return out;
}

int BatchEngine::sync() {
  UBG_HIP(hipStreamSynchronize(stream_));
  return UBG_OK;
}

int BatchEngine::set_tuning(const Tuning &t) {
  tune_ = t;
  drop_graphs();
  const int rc = build_tiles();
  if (rc != UBG_OK) invalidate_members(); // the tile maps are the former tuning's
  return rc;
}

// nu_pre sweeps of every member level, `reps` times (scratch buffers only:
// the next update zeroes e before it is used)
int BatchEngine::launch_sweeps_only(int reps) {
  const int n = (int)all_.size();
  std::vector<uint8_t> idx(2 * (size_t)n, 0);
  uint8_t *d_idx = nullptr;
  UBG_TRY(upload_idx(idx, &d_idx));
  for (int r = 0; r < reps; r++)
    for (int l = 0; l < lmax_; l++) {
      if (!sw_[l].n) continue;
      StageArgs a{};
      a.lev = d_lev_;
      a.dom = d_dom_;
      a.level = l;
      a.ia = d_idx;
      a.ib = d_idx + n;
      a.alpha = prm_.alpha;
      a.off = d_off_ + sw_[l].off;
      a.ndom = sw_[l].nd;
      a.ntiles = sw_[l].n;
      int b = tune_.blocks > 0 ? std::min(a.ntiles, tune_.blocks) : a.ntiles;
      launch_sweep(tune_, std::max(b, 1), stream_, a);
    }
  UBG_TRY(check_launch());
  return UBG_OK;
}

// the pre passes of every member level, then the post passes, `reps`
// times (scratch buffers only, as launch_sweeps_only)
int BatchEngine::launch_passes_only(int reps) {
  const int n = (int)all_.size();
  std::vector<uint8_t> idx(2 * (size_t)n, 0);
  uint8_t *d_idx = nullptr;
  UBG_TRY(upload_idx(idx, &d_idx));
  auto pass = [&](bool pre, int l) {
    const Span &sp = pre ? tp_[l] : tq_[l];
    if (!sp.n) return;
    StageArgs a{};
    a.lev = d_lev_;
    a.dom = d_dom_;
    a.level = l;
    a.ia = d_idx;
    a.ib = d_idx + n;
    a.alpha = prm_.alpha;
    a.off = d_off_ + sp.off;
    a.ndom = sp.nd;
    a.ntiles = sp.n;
    a.oty = sp.oty;
    int b = tune_.blocks > 0 ? std::min(a.ntiles, tune_.blocks) : a.ntiles;
    launch_batch_pass(sp.shape, pre, pre ? prm_.nu_pre : prm_.nu_post, false, std::max(b, 1),
                      stream_, a);
  };
  for (int r = 0; r < reps; r++) {
    for (int l = 0; l < lmax_; l++) pass(true, l);
    for (int l = lmax_ - 1; l >= 0; l--) pass(false, l);
  }
  UBG_TRY(check_launch());
  return UBG_OK;
}

// Times the candidate shapes over the member levels and keeps the fastest:
// the level passes' tile shapes x block counts when the levels run as
// passes, else the smoother tile shapes x block counts.
int BatchEngine::autotune(double *best_ms) {
  const Tuning saved = tune_;
  Tuning best = saved;
  double best_t = 1e30;
  hipEvent_t e0, e1;
  UBG_HIP(hipEventCreate(&e0));
  UBG_HIP(hipEventCreate(&e1));
  const int block_opts[] = {0, 2048, 1024};
  std::vector<Tuning> cand;
  if (tiled()) {
    for (int r : {0, 8, 16, 32})
      for (int bo : block_opts) cand.push_back(Tuning{saved.tx, saved.ty, bo, r});
  } else {
    for (const Shape &sh : kShapes)
      for (int bo : block_opts) cand.push_back(Tuning{sh.tx, sh.ty, bo, saved.prow});
  }
  // the solve state must allow the sweeps: mark members active meanwhile
  std::vector<DState> st(all_.size());
  for (size_t i = 0; i < all_.size(); i++) UBG_TRY(domain_read_state(all_[i], &st[i]));
  for (size_t i = 0; i < all_.size(); i++) {
    DState s = st[i];
    s.active = 1;
    UBG_HIP(hipMemcpyAsync(all_[i]->st, &s, sizeof(s), hipMemcpyHostToDevice, stream_));
  }
  int rc = UBG_OK;
  for (const Tuning &c : cand) {
    tune_ = c;
    if ((rc = build_tiles()) != UBG_OK) break;
    auto run = [&](int reps) { return tiled() ? launch_passes_only(reps) : launch_sweeps_only(reps); };
    if ((rc = run(1)) != UBG_OK) break; // warm
    (void)hipEventRecord(e0, stream_);
    if ((rc = run(3)) != UBG_OK) break;
    (void)hipEventRecord(e1, stream_);
    (void)hipEventSynchronize(e1);
    float ms = 0.0f;
    (void)hipEventElapsedTime(&ms, e0, e1);
    if (ms < best_t) {
      best_t = ms;
      best = tune_;
    }
  }
  for (size_t i = 0; i < all_.size(); i++)
    (void)hipMemcpyAsync(all_[i]->st, &st[i], sizeof(DState), hipMemcpyHostToDevice, stream_);
  (void)hipStreamSynchronize(stream_);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  const int rt = set_tuning(rc == UBG_OK ? best : saved);
  if (best_ms) *best_ms = best_t / 3.0;
  return rc != UBG_OK ? rc : rt;
}

} // namespace ubg

// ===========================================================================
// C ABI: ubg_batch
// ===========================================================================
struct ubg_batch {
  ubg::BatchEngine eng;
  ubg::Arena arena;
  hipStream_t stream = nullptr;
  std::vector<ubg::BDomain *> doms;
  std::vector<int> ws, hs;
  std::vector<bool> ready;
  std::recursive_mutex mu;
  // projection solves: every domain's solve state is active (refinement
  // solves end domains; the next projection re-activates them)
  bool proj_active = false;
  // batched simulation steps: the simulation and flag generation each
  // domain's geometry was built from, and the events that order the
  // simulations' streams around the batch's
  std::vector<const ubg_sim *> src;
  std::vector<unsigned> src_gen;
  std::vector<hipEvent_t> ev_ready;
  std::shared_ptr<ubg::ExtEvent> ev_done; // recorded after each batched step
  // the per-stage simulation tables of a batched step: two slots used in
  // turn (pinned staging and device copy), each free again once its event
  // has passed
  struct TabSlot {
    ubg::SimRec *host = nullptr, *dev = nullptr;
    size_t cap = 0;
    hipEvent_t used = nullptr;
  } slot[2];
  int next_slot = 0;
};

namespace {

int batch_check(ubg_batch *b, int d) {
  if (!b) return fail(UBG_E_INVALID, "null batch");
  if (d < 0 || d >= (int)b->ws.size()) return fail(UBG_E_INVALID, "domain index out of range");
  return UBG_OK;
}

// The kernels that a line of a tuning file was timed with: counted up when its
// numbers come to name other ones (2: pass_rows names shapes of register
// tiles, before that rows of LDS tiles), so that an older line is timed anew.
constexpr uint64_t kTuningKernels = 2;
std::string batch_key(const ubg_batch *b, const ubg_params &p, int k) {
  // FNV-1a over the sizes, the smoothing counts, alpha (off 1 no row takes the
  // uniform update) and the kernels
  uint64_t hsh = 1469598103934665603ull;
  auto mix = [&](uint64_t v) {
    for (int i = 0; i < 8; i++) {
      hsh ^= (v >> (8 * i)) & 0xff;
      hsh *= 1099511628211ull;
    }
  };
  for (size_t i = 0; i < b->ws.size(); i++) {
    mix((uint64_t)b->ws[i]);
    mix((uint64_t)b->hs[i]);
  }
  mix((uint64_t)p.nu_pre);
  mix((uint64_t)p.nu_post);
  mix((uint64_t)p.nu_coarse);
  mix((uint64_t)k);
  uint32_t alpha;
  std::memcpy(&alpha, &p.alpha, sizeof alpha);
  mix(alpha);
  mix(kTuningKernels);
  char buf[40];
  std::snprintf(buf, sizeof(buf), "%016llx", (unsigned long long)hsh);
  return buf;
}

} // namespace

extern "C" {

UBG_API int ubg_batch_bytes(int n, const int *widths, const int *heights, size_t *bytes) {
  if (n <= 0 || !widths || !heights || !bytes) return fail(UBG_E_INVALID, "bad arguments");
  size_t tot = 0;
  for (int i = 0; i < n; i++) {
    ubg::BShape s;
    UBG_TRY(ubg::batch_shape(widths[i], heights[i], &s));
    tot += s.geom_bytes + s.dom_bytes;
  }
  *bytes = tot;
  return UBG_OK;
}

UBG_API int ubg_batch_create(int n, const int *widths, const int *heights, const ubg_params *prm,
                             ubg_batch **out) {
  if (!out) return fail(UBG_E_INVALID, "null output pointer");
  int nd = 0;
  ubg_device_count(&nd);
  if (nd <= 0) return fail(UBG_E_NO_DEVICE, "no HIP device visible");
  size_t bytes = 0;
  UBG_TRY(ubg_batch_bytes(n, widths, heights, &bytes));
  ubg_params P;
  default_params(&P);
  if (prm) {
    UBG_TRY(check_params(prm));
    P = *prm;
  }
  auto *b = new ubg_batch();
  hipError_t e = hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking);
  if (e != hipSuccess) {
    delete b;
    return fail(UBG_E_HIP, std::string("hipStreamCreate: ") + hipGetErrorString(e));
  }
  b->ws.assign(widths, widths + n);
  b->hs.assign(heights, heights + n);
  b->ready.assign(n, false);
  b->doms.assign(n, nullptr);
  int rc = b->arena.init(bytes + 4096);
  if (rc == UBG_OK) rc = b->eng.init(b->stream, P, 4, n);
  if (rc != UBG_OK) {
    ubg_batch_destroy(b);
    return rc;
  }
  *out = b;
  return UBG_OK;
}

UBG_API int ubg_batch_destroy(ubg_batch *b) {
  if (!b) return UBG_OK;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  for (auto *d : b->doms)
    if (d) b->eng.domain_release(b->arena, d);
  b->doms.clear();
  b->arena.release();
  for (hipEvent_t e : b->ev_ready)
    if (e) (void)hipEventDestroy(e);
  for (auto &t : b->slot) {
    if (t.host) (void)hipHostFree(t.host);
    if (t.dev) (void)hipFree(t.dev);
    if (t.used) (void)hipEventDestroy(t.used);
  }
  hipStream_t s = b->stream;
  delete b; // the engine frees its tables first
  if (s) (void)hipStreamDestroy(s);
  return UBG_OK;
}

namespace {

int set_domain(ubg_batch *b, int d, const float *flag, const float *rhs, float h, bool need_ring) {
  UBG_TRY(batch_check(b, d));
  if (!flag || !rhs) return fail(UBG_E_INVALID, "null argument");
  if (!(h > 0.0f) || !std::isfinite(h)) return fail(UBG_E_INVALID, "h must be positive");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  if (b->doms[d]) {
    b->eng.invalidate_members();
    b->eng.domain_release(b->arena, b->doms[d]);
    b->doms[d] = nullptr;
  }
  ubg::BGeom *geo = nullptr;
  UBG_TRY(b->eng.geom_create(b->arena, b->ws[d], b->hs[d], flag, &geo, need_ring));
  ubg::BDomain *dom = nullptr;
  int rc = b->eng.domain_create(b->arena, geo, h, &dom);
  b->eng.geom_release(b->arena, geo); // the domain holds its reference
  if (rc) return rc;
  b->doms[d] = dom;
  b->proj_active = false;
  rc = b->eng.domain_set_rhs(dom, rhs);
  b->ready[d] = rc == UBG_OK;
  return rc;
}

} // namespace

UBG_API int ubg_batch_set_domain(ubg_batch *b, int d, const float *flag, const float *rhs, float h) {
  return set_domain(b, d, flag, rhs, h, true);
}

UBG_API int ubg_batch_set_projection_domain(ubg_batch *b, int d, const float *flag,
                                            const float *rhs, float h) {
  return set_domain(b, d, flag, rhs, h, false);
}

UBG_API int ubg_batch_set_rhs(ubg_batch *b, int d, const float *rhs) {
  UBG_TRY(batch_check(b, d));
  if (!rhs) return fail(UBG_E_INVALID, "null argument");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  if (!b->doms[d]) return fail(UBG_E_STATE, "domain not set");
  return b->eng.domain_set_rhs(b->doms[d], rhs);
}

UBG_API int ubg_batch_set_guess(ubg_batch *b, int d, const double *x) {
  UBG_TRY(batch_check(b, d));
  std::lock_guard<std::recursive_mutex> g(b->mu);
  if (!b->doms[d]) return fail(UBG_E_STATE, "domain not set");
  return b->eng.domain_set_guess(b->doms[d], x);
}

UBG_API int ubg_batch_set_pressure(ubg_batch *b, int d, const float *p) {
  UBG_TRY(batch_check(b, d));
  std::lock_guard<std::recursive_mutex> g(b->mu);
  if (!b->doms[d]) return fail(UBG_E_STATE, "domain not set");
  if (p) {
    const size_t n = (size_t)b->ws[d] * b->hs[d];
    for (size_t i = 0; i < n; i++)
      if (!std::isfinite(p[i])) return fail(UBG_E_NONFINITE, "pressure has a non-finite value");
  }
  return b->eng.domain_set_level0(b->doms[d], p, nullptr, hipMemcpyHostToDevice);
}

UBG_API int ubg_batch_get_pressure(ubg_batch *b, int d, float *p) {
  UBG_TRY(batch_check(b, d));
  if (!p) return fail(UBG_E_INVALID, "null output");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  if (!b->doms[d]) return fail(UBG_E_STATE, "domain not set");
  return b->eng.domain_get_pressure(b->doms[d], p, hipMemcpyDeviceToHost);
}

namespace {

// every domain a running member with an active solve state
int proj_members(ubg_batch *b) {
  if (!b->proj_active) {
    for (auto *d : b->doms) UBG_TRY(b->eng.domain_start(d, 0.5, 1));
    b->proj_active = true;
  }
  return b->eng.set_members(b->doms, {});
}

} // namespace

UBG_API int ubg_batch_vcycles(ubg_batch *b, int ncycles, int zero_gradient_bc) {
  if (!b) return fail(UBG_E_INVALID, "null batch");
  if (ncycles < 1 || ncycles > 1000) return fail(UBG_E_INVALID, "ncycles must be in 1..1000");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  for (size_t i = 0; i < b->doms.size(); i++)
    if (!b->ready[i]) return fail(UBG_E_STATE, "domain " + std::to_string(i) + " not set");
  // the level-0 rhs of the V-cycles is the domain's rhs
  for (auto *d : b->doms)
    UBG_HIP(hipMemcpyAsync(d->f[0], d->rhs, (size_t)d->g->W * d->g->H * 4,
                           hipMemcpyDeviceToDevice, b->stream));
  UBG_TRY(proj_members(b));
  UBG_TRY(b->eng.enqueue_vcycles(ncycles, zero_gradient_bc != 0));
  UBG_HIP(hipStreamSynchronize(b->stream));
  return check_launch();
}

namespace {

// the copies of `jobs`, kCopyJobs per launch
int launch_copies(const std::vector<ubg::CopyJob> &jobs, hipStream_t s) {
  for (size_t b = 0; b < jobs.size(); b += ubg::kCopyJobs) {
    ubg::CopyJobs cj{};
    const int nj = (int)std::min<size_t>(ubg::kCopyJobs, jobs.size() - b);
    int maxn = 0;
    for (int k = 0; k < nj; k++) {
      cj.j[k] = jobs[b + k];
      maxn = std::max(maxn, cj.j[k].n);
    }
    const int gx = std::max(1, std::min((maxn + 1023) / 1024, 512));
    hipLaunchKernelGGL(ubg::kb_copy_level0, dim3(gx, nj), dim3(256), 0, s, cj, nj);
  }
  return check_launch();
}

bool same_solver(const ubg_params &a, const ubg_params &b) {
  return a.nu_pre == b.nu_pre && a.nu_post == b.nu_post && a.nu_coarse == b.nu_coarse &&
         a.vcycles_per_step == b.vcycles_per_step && a.alpha == b.alpha;
}

// whether a simulation appears more than once in the list (one batched
// step would then advance its fields twice in the same launches)
bool repeats(ubg_sim *const *sims, int n) {
  std::vector<ubg_sim *> v(sims, sims + n);
  std::sort(v.begin(), v.end());
  return std::adjacent_find(v.begin(), v.end()) != v.end();
}

// (re)build domain d from simulation s's level-0 flag and h
int domain_from_sim(ubg_batch *b, int d, ubg_sim *s) {
  const ubg::SimLevel0 q = ubg::sim_level0(s);
  const size_t n = (size_t)q.W * q.H;
  std::vector<uint8_t> fl(n);
  UBG_HIP(hipStreamSynchronize(q.stream));
  UBG_HIP(hipMemcpy(fl.data(), q.flag, n, hipMemcpyDeviceToHost));
  std::vector<float> flag(n), zero(n, 0.0f);
  for (size_t i = 0; i < n; i++) flag[i] = fl[i] ? 1.0f : 0.0f;
  UBG_TRY(ubg_batch_set_projection_domain(b, d, flag.data(), zero.data(), q.h));
  b->src[d] = s;
  b->src_gen[d] = q.flag_gen;
  b->proj_active = false;
  return UBG_OK;
}

} // namespace

UBG_API int ubg_batch_create_for_sims(ubg_sim *const *sims, int n, ubg_batch **out) {
  if (!sims || !out || n < 1) return fail(UBG_E_INVALID, "null argument or n < 1");
  std::vector<int> ws(n), hs(n);
  ubg_params prm{};
  for (int i = 0; i < n; i++) {
    if (!sims[i]) return fail(UBG_E_INVALID, "null simulation");
    const ubg::SimLevel0 q = ubg::sim_level0(sims[i]);
    if (i == 0) prm = q.prm;
    else if (!same_solver(prm, q.prm))
      return fail(UBG_E_INVALID, "the simulations' multigrid parameters differ");
    ws[i] = q.W;
    hs[i] = q.H;
  }
  if (repeats(sims, n)) return fail(UBG_E_INVALID, "a simulation appears twice in the list");
  ubg_batch *b = nullptr;
  UBG_TRY(ubg_batch_create(n, ws.data(), hs.data(), &prm, &b));
  b->src.assign(n, nullptr);
  b->src_gen.assign(n, 0u);
  for (int i = 0; i < n; i++) {
    const int rc = domain_from_sim(b, i, sims[i]);
    if (rc != UBG_OK) {
      ubg_batch_destroy(b);
      return rc;
    }
  }
  *out = b;
  return UBG_OK;
}

UBG_API int ubg_sims_step(ubg_batch *b, ubg_sim *const *sims, int n, const float *dts) {
  if (!b || !sims || !dts) return fail(UBG_E_INVALID, "null argument");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  if (n != (int)b->doms.size() || b->src.size() != b->doms.size())
    return fail(UBG_E_INVALID, "the batch was not made for these simulations");
  const ubg_params &bp = b->eng.params();
  std::vector<ubg::SimLevel0> q(n);
  for (int i = 0; i < n; i++) {
    if (!sims[i]) return fail(UBG_E_INVALID, "null simulation");
    q[i] = ubg::sim_level0(sims[i]);
    if (q[i].W != b->ws[i] || q[i].H != b->hs[i] || !same_solver(bp, q[i].prm))
      return fail(UBG_E_INVALID, "simulation " + std::to_string(i) + " does not match its domain");
    if (!std::isfinite(dts[i])) return fail(UBG_E_INVALID, "dt is not finite");
  }
  if (repeats(sims, n)) return fail(UBG_E_INVALID, "a simulation appears twice in the list");
  // geometry of a domain whose simulation changed its flags (or is another one)
  for (int i = 0; i < n; i++)
    if (b->src[i] != sims[i] || b->src_gen[i] != q[i].flag_gen) {
      UBG_TRY(domain_from_sim(b, i, sims[i]));
      q[i] = ubg::sim_level0(sims[i]);
    }
  if (!b->ev_done) {
    auto e = std::make_shared<ubg::ExtEvent>();
    UBG_HIP(hipEventCreateWithFlags(&e->ev, hipEventDisableTiming));
    b->ev_done = e;
  }
  while ((int)b->ev_ready.size() < n) {
    hipEvent_t e = nullptr;
    UBG_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    b->ev_ready.push_back(e);
  }
  // a free table slot (allocated before any simulation's state moves)
  auto &T = b->slot[b->next_slot];
  b->next_slot ^= 1;
  const size_t nt = (size_t)4 * n;
  if (!T.used) UBG_HIP(hipEventCreateWithFlags(&T.used, hipEventDisableTiming));
  UBG_HIP(hipEventSynchronize(T.used)); // the step two calls ago has read it
  if (T.cap < nt) {
    if (T.host) (void)hipHostFree(T.host);
    if (T.dev) (void)hipFree(T.dev);
    T.host = nullptr;
    T.dev = nullptr;
    T.cap = 0;
    UBG_HIP(hipHostMalloc((void **)&T.host, nt * sizeof(ubg::SimRec), hipHostMallocDefault));
    UBG_HIP(hipMalloc((void **)&T.dev, nt * sizeof(ubg::SimRec)));
    T.cap = nt;
  }
  // The per-cell stages of every simulation's step as records (their
  // applyAccumulatedVelocity / boundary / face-factor preludes, when due,
  // run on the simulations' own streams); the batch's stream then waits for
  // every simulation whose stream had work of its own since the last step.
  std::vector<ubg::SimRec> rec((size_t)4 * n);
  std::vector<char> sinks(n, 0);
  for (int i = 0; i < n; i++) {
    bool has = false;
    UBG_TRY(ubg::sim_batched_records(sims[i], dts[i], &rec[(size_t)4 * i], &has));
    sinks[i] = has;
  }
  for (int i = 0; i < n; i++)
    if (ubg::sim_take_own_work(sims[i])) {
      UBG_HIP(hipEventRecord(b->ev_ready[i], q[i].stream));
      UBG_HIP(hipStreamWaitEvent(b->stream, b->ev_ready[i], 0));
    }
  // stage tables: stage k of simulation i at [k n + i], rows numbered
  // through the simulations' interiors
  int rows = 0, maxw = 0;
  bool buf = true;
  for (int i = 0; i < n; i++) {
    for (int k = 0; k < 4; k++) {
      ubg::SimRec r = rec[(size_t)4 * i + k];
      r.row0 = rows;
      T.host[(size_t)k * n + i] = r;
    }
    rows += q[i].H - 2;
    maxw = std::max(maxw, q[i].W);
    buf = buf && (size_t)q[i].W * q[i].H * 4 < ((size_t)1 << 31);
  }
  UBG_HIP(hipMemcpyAsync(T.dev, T.host, nt * sizeof(ubg::SimRec), hipMemcpyHostToDevice, b->stream));
  const ubg::SimRec *tab = T.dev;
  // diffuse (two iterations), advect, setVBCs + divergence of all
  // simulations, one launch each; sinks stamped in list order after the
  // divergence
  ubg::launch_sims_diffuse(tab, n, rows, maxw, b->stream);
  ubg::launch_sims_diffuse(tab + n, n, rows, maxw, b->stream);
  ubg::launch_sims_advect(tab + 2 * n, n, rows, maxw, buf, b->stream);
  ubg::launch_sims_vbcs_divergence(tab + 3 * n, n, rows, maxw, b->stream);
  UBG_TRY(check_launch());
  for (int i = 0; i < n; i++)
    if (sinks[i]) UBG_TRY(ubg::sim_apply_sinks_on(sims[i], b->stream));
  // the V-cycles of all of them (the level-0 pressure and rhs gathered in
  // one launch, the pressure scattered back in another)
  UBG_TRY(proj_members(b));
  std::vector<ubg::CopyJob> in(n), out(n);
  for (int i = 0; i < n; i++) {
    ubg::BDomain *d = b->doms[i];
    in[i] = ubg::CopyJob{q[i].p, q[i].f, d->p[0][d->cur[0]], d->f[0], q[i].W * q[i].H};
  }
  UBG_TRY(launch_copies(in, b->stream));
  UBG_TRY(b->eng.enqueue_vcycles(bp.vcycles_per_step, true));
  for (int i = 0; i < n; i++) {
    ubg::BDomain *d = b->doms[i];
    out[i] = ubg::CopyJob{d->p[0][d->cur[0]], nullptr, q[i].p, nullptr, q[i].W * q[i].H};
  }
  UBG_TRY(launch_copies(out, b->stream));
  // setPBC + correction + setVBCs + saveCurrent of all of them
  ubg::launch_sims_correct_tail(tab + 3 * n, n, rows, maxw, b->stream);
  UBG_TRY(check_launch());
  UBG_HIP(hipEventRecord(T.used, b->stream));
  // each simulation's next own work waits for this step
  UBG_HIP(hipEventRecord(b->ev_done->ev, b->stream));
  for (int i = 0; i < n; i++) ubg::sim_set_ext_event(sims[i], b->ev_done);
  return UBG_OK;
}

UBG_API int ubg_batch_solve(ubg_batch *b, const ubg_ir_params *prm, int *graph_replays) {
  if (!b) return fail(UBG_E_INVALID, "null batch");
  ubg_ir_params P;
  ubg_ir_params_default(&P);
  if (prm) P = *prm;
  if (!(P.tol > 0.0 && P.tol < 1.0)) return fail(UBG_E_INVALID, "tol must be in (0, 1)");
  if (P.vcycles_per_iter < 1 || P.vcycles_per_iter > 256 || P.max_iter < 1 || P.max_iter > 1000000)
    return fail(UBG_E_INVALID, "vcycles_per_iter or max_iter out of range");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  for (size_t i = 0; i < b->doms.size(); i++) {
    if (!b->ready[i]) return fail(UBG_E_STATE, "domain " + std::to_string(i) + " not set");
    if (!b->doms[i]->g->ring_fluid)
      return fail(UBG_E_FLAG_VALUE, "domain " + std::to_string(i) +
                                        " has a solid outer-ring cell: projection solves only");
  }
  b->eng.set_vcycles(P.vcycles_per_iter);
  b->proj_active = false;
  UBG_TRY(b->eng.start_all(b->doms, P.tol, P.max_iter));
  // first update of every domain (r0), then rounds of two steps
  UBG_TRY(b->eng.set_members(b->doms, {}));
  UBG_TRY(b->eng.enqueue_first_update());
  UBG_TRY(b->eng.sync());
  // when domains finish, shrink the member set to the active ones (new tables
  // and tiles) so finished domains cost no dispatch.  A round's launches (2 to
  // 3 us of host time each) run ahead of its kernels (5 us and more), and the
  // tables of a new member set are uploaded without waiting; a graph captured
  // and instantiated per member set, over tables copied with two
  // synchronisations, left the GPU idle meanwhile: 24 domains of 128 to 1024
  // cells a side 10.1 -> 7.9 ms, 60 of 100x90 to 513x385 14.4 -> 10.2 ms, one
  // domain the same (256x200: 2.73 and 2.75 ms).  Only a batch of one domain with
  // a launch per sweep runs its launches faster than they are enqueued, and its
  // member set stays: replayed (64x64 at 20 sweeps 1.83 -> 1.69 ms, 256x200 6.2
  // -> 5.5; two domains of 48x48 the other way round, 2.7 and 3.7, for a graph
  // of the one that is left).
  const bool lone_sweeps = b->doms.size() == 1 && !b->eng.tiled();
  int rounds = 0;
  while (b->eng.active_count() > 0 && 2 * rounds < P.max_iter + 2) {
    std::vector<ubg::BDomain *> act = b->eng.active_members();
    if (act.size() != b->eng.members()) UBG_TRY(b->eng.set_members(act, {}));
    UBG_TRY(lone_sweeps ? b->eng.replay_steps(2) : b->eng.enqueue_steps(2));
    UBG_TRY(b->eng.sync());
    rounds++;
  }
  if (graph_replays) *graph_replays = rounds;
  int bad = 0;
  std::vector<ubg::DState> states;
  UBG_TRY(b->eng.read_states(b->doms, states));
  for (size_t i = 0; i < b->doms.size(); i++) {
    const ubg::DState &s = states[i];
    b->doms[i]->xcur = s.xcur;
    if (s.nonfinite) return fail(UBG_E_NONFINITE, "a domain's residual is not finite");
    if (!s.converged) bad++;
  }
  if (bad)
    return fail(UBG_E_NOT_CONVERGED, std::to_string(bad) + " domain(s) stopped short of tol");
  return UBG_OK;
}

UBG_API int ubg_batch_result(ubg_batch *b, int d, ubg_ir_result *res) {
  UBG_TRY(batch_check(b, d));
  if (!res) return fail(UBG_E_INVALID, "null result");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  if (!b->doms[d]) return fail(UBG_E_STATE, "domain not set");
  ubg::DState s;
  UBG_TRY(b->eng.domain_read_state(b->doms[d], &s));
  std::memset(res, 0, sizeof(*res));
  res->iterations = s.iters;
  res->vcycles = s.vcycles;
  res->converged = s.converged;
  res->r0_norm = s.r0;
  res->rel_residual = s.rel;
  for (int i = 0; i < std::min(s.iters, UBG_IR_HISTORY); i++) res->history[i] = s.hist[i];
  return UBG_OK;
}

UBG_API int ubg_batch_get_solution(ubg_batch *b, int d, double *x) {
  UBG_TRY(batch_check(b, d));
  if (!x) return fail(UBG_E_INVALID, "null destination");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  if (!b->doms[d]) return fail(UBG_E_STATE, "domain not set");
  return b->eng.domain_get_solution(b->doms[d], x);
}

UBG_API int ubg_batch_set_tuning(ubg_batch *b, const ubg_batch_tuning *t) {
  if (!b || !t) return fail(UBG_E_INVALID, "null argument");
  if (!shape_ok(t->tile_w, t->tile_h)) return fail(UBG_E_INVALID, "tile shape not compiled");
  if (t->blocks < 0) return fail(UBG_E_INVALID, "negative block count");
  const int rows = t->pass_rows;
  if (!pass_rows_ok(rows)) return fail(UBG_E_INVALID, "pass_rows must be 0, 8, 16 or 32");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  return b->eng.set_tuning(ubg::Tuning{t->tile_w, t->tile_h, t->blocks, rows});
}

UBG_API int ubg_batch_get_tuning(ubg_batch *b, ubg_batch_tuning *t) {
  if (!b || !t) return fail(UBG_E_INVALID, "null argument");
  const ubg::Tuning &x = b->eng.tuning();
  t->tile_w = x.tx;
  t->tile_h = x.ty;
  t->blocks = x.blocks;
  t->pass_rows = x.prow;
  t->sweep_ms = 0.0;
  return UBG_OK;
}

UBG_API int ubg_batch_autotune(ubg_batch *b, const char *db_path, ubg_batch_tuning *out) {
  if (!b) return fail(UBG_E_INVALID, "null batch");
  std::lock_guard<std::recursive_mutex> g(b->mu);
  for (size_t i = 0; i < b->doms.size(); i++)
    if (!b->ready[i]) return fail(UBG_E_STATE, "domain " + std::to_string(i) + " not set");
  const std::string key = batch_key(b, b->eng.params(), b->eng.vcycles());
  if (db_path) {
    std::ifstream in(db_path);
    std::string line;
    while (std::getline(in, line)) {
      std::istringstream ls(line);
      std::string k;
      int tx, ty, bl, rows;
      double ms;
      if (ls >> k >> tx >> ty >> bl >> rows >> ms && k == key && shape_ok(tx, ty) && bl >= 0 &&
          pass_rows_ok(rows)) {
        UBG_TRY(b->eng.set_tuning(ubg::Tuning{tx, ty, bl, rows}));
        if (out) *out = ubg_batch_tuning{tx, ty, bl, rows, ms};
        return UBG_OK;
      }
    }
  }
  UBG_TRY(b->eng.set_members(b->doms, {}));
  double ms = 0.0;
  UBG_TRY(b->eng.autotune(&ms));
  const ubg::Tuning &t = b->eng.tuning();
  if (out) *out = ubg_batch_tuning{t.tx, t.ty, t.blocks, t.prow, ms};
  if (db_path) {
    std::ofstream o(db_path, std::ios::app);
    if (!o) return fail(UBG_E_INVALID, std::string("cannot write tuning db ") + db_path);
    o << key << " " << t.tx << " " << t.ty << " " << t.blocks << " " << t.prow << " " << ms << "\n";
  }
  return UBG_OK;
}

} // extern "C"
