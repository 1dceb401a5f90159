// coarse_device.hpp -- the single-workgroup LDS V-cycle of the coarse
// levels (MG::solveLevel, pressure_solver.cpp:201-248, from a level whose
// whole sub-hierarchy fits in LDS down to the coarsest solved level L-2),
// shared by the single-domain and the batched solvers.
#pragma once

#include "mg_device.hpp"

namespace ubg {

constexpr int MAXL = 16;
constexpr int TPB_C = 1024;
constexpr int WAVES_C = TPB_C / 64;
constexpr size_t LDS_BUDGET = 152 * 1024;
// The single-workgroup LDS V-cycle starts at the first level with at most
// this many cells: one CU does all of its work, so larger levels run faster as
// tiles spread over the chip (128x64 and below in LDS at 3/3/5 sweeps: 32 us,
// against 12.5 us from 64x32 and 12.6 us for the tiles of 128x64).
constexpr size_t kCoarseMaxCells = 4096;

struct CoarseArgs {
  int n; // levels first .. L-2
  int w[MAXL], h[MAXL];
  float hh[MAXL];
  float ihsq[MAXL]; // 1 / h / h
  float iw[MAXL];   // 1 / w
  int op[MAXL], of[MAXL], om[MAXL]; // LDS byte offsets of p, f, mask
  int orr;                           // residual scratch (first level's size)
  const uint8_t *mask[MAXL];
  const float *f0;
  float *p0;
  int nu_pre, nu_post, nu_coarse;
  float alpha;
};

// Threads own pairs of cells: thread t has pair t, t + 1024, ... of a level,
// pair t being the cells 2t and 2t + 1 in row-major order -- one red
// ((x + y) odd) and one black, neighbours in a row (or, at an odd width, two
// ring cells of adjacent rows).  For a visit of the level the pair's p, f and
// decoded smoothing rules stay in registers (the first level's for the whole
// V-cycle).  LDS holds p for the neighbours, the red cells and the black ones
// each in a plane of their own, entry i >> 1 for cell i: a colour reads only
// the other plane, and a wave's lanes read consecutive words.  An update is
// three LDS reads (its partner is a register) and one write.
//
// What bounds this kernel is latency and the instructions of one CU: about
// 35 dependent colour phases and two grid transfers per pair of levels.
// Measured on gfx950 (64x32 down to 16x8, 3/3/5 sweeps; 64x64 down to 8x8):
// 12.4 and 19.7 us, against 15.2 and 27.4 us with one cell per
// thread and phase in row-major LDS, whose transfers alone cost 3.2 us per
// pair of levels (integer divisions, idle waves at work, two-way bank
// conflicts in every phase).
//
// A cell's smoothing constants, decoded from its mask byte and f.  smooth_rule
// performs the operations of smooth() (the division by the count as div_count
// does it); the first two addends, W and E, are its outside and its partner
// neighbour in either order, which rounds alike.
struct CellRule {
  int so, sp, ss, sn; // 0 / -1: the neighbour's value is kept, or +0 added
  float inv, ns;      // RN(1 / s) and -s for the neighbour count s
  float F, fhh;       // own flag (0 / 1) and (f * h) * h
  int some;           // 0 when s == 0 (the quotient is +0), else -1
};
__device__ __forceinline__ CellRule cell_rule(unsigned mk, bool out_west, float fv, float h) {
  CellRule c;
  const int sw = -(int)((mk >> 1) & 1u), se = -(int)((mk >> 2) & 1u);
  c.so = out_west ? sw : se;
  c.sp = out_west ? se : sw;
  c.ss = -(int)((mk >> 3) & 1u);
  c.sn = -(int)((mk >> 4) & 1u);
  const unsigned s = mk >> 5;
  const float pow2 = __int_as_float((int)((127u - (s >> 1)) << 23));
  c.inv = (s == 3u) ? (1.0f / 3.0f) : pow2;
  c.ns = -(float)s;
  c.some = s == 0u ? 0 : -1;
  c.F = (float)(mk & MK_SELF);
  c.fhh = fv * h * h;
  return c;
}
__device__ __forceinline__ float keep(int sel, float v) {
  return __int_as_float(__float_as_int(v) & sel);
}
__device__ __forceinline__ float pick(int sel, float v, float c) {
  return __int_as_float((__float_as_int(v) & sel) | (__float_as_int(c) & ~sel));
}
__device__ __forceinline__ float smooth_rule(float pc, float po, float pp, float ps, float pn,
                                             const CellRule &c, float alpha) {
  float val = 0.0f;
  val += keep(c.so, po);
  val += keep(c.sp, pp);
  val += keep(c.ss, ps);
  val += keep(c.sn, pn);
  val += c.fhh;
  const float q = val * c.inv;
  const float r = fmaf(c.ns, q, val);
  const float q2 = fmaf(r, c.inv, q);
  val = keep(c.some, q2);
  return c.F * (alpha * val + (1.0f - alpha) * pc);
}
// residual_of with the rule's selectors (f itself beside the rule)
__device__ __forceinline__ float residual_rule(float pc, float po, float pp, float ps, float pn,
                                               float fv, const CellRule &c, float ihsq) {
  float val = 0.0f;
  val += pick(c.so, po, pc);
  val += pick(c.sp, pp, pc);
  val += pick(c.ss, ps, pc);
  val += pick(c.sn, pn, pc);
  val += -4.0f * pc;
  val *= ihsq;
  return c.F != 0.0f ? fv + val : 0.0f;
}

// flag count + the double literal 0.0001, stored as float (pressure_solver.cpp:149)
__device__ __forceinline__ float eps_sum(int s) { return (float)((double)s + 0.0001); }

// one level in LDS; planes: red at [0], black at [half]
struct LdsLevel {
  float *P, *Fv;
  uint8_t *M;
  int w, h, n, half; // cells, entries of a plane (= pairs)
  float hh, ihsq, iw;
  // row of cell i: (i + 1/2) / w is at least 1 / (2 w) from an integer, more
  // than the product's rounding error for any i in LDS
  __device__ __forceinline__ int row_of(int i) const { return (int)(((float)i + 0.5f) * iw); }
  __device__ __forceinline__ float *plane(float *base, int black) const {
    return base + (black ? half : 0);
  }
};
__device__ __forceinline__ LdsLevel lds_level(const CoarseArgs &a, char *smem, int l) {
  LdsLevel L;
  L.P = (float *)(smem + a.op[l]);
  L.Fv = (float *)(smem + a.of[l]);
  L.M = (uint8_t *)(smem + a.om[l]);
  L.w = a.w[l];
  L.h = a.h[l];
  L.n = L.w * L.h;
  L.half = (L.n + 1) >> 1;
  L.hh = a.hh[l];
  L.ihsq = a.ihsq[l];
  L.iw = a.iw[l];
  return L;
}

// ordering of a phase's LDS writes before the next phase's reads: a level
// whose pairs all belong to one wave needs no barrier (a wave's LDS
// operations execute in order)
__device__ __forceinline__ void phase_end(bool one_wave) {
  if (one_wave) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  else __syncthreads();
}

// The thread's K pairs of a level.  r: the pair's red cell, b: its black one.
template <int K> struct LevelPairs {
  int t[K], i0[K];                // pair, its first cell
  int x0[K], y0[K];               // column and row of the first cell
  bool rfirst[K];                 // the first cell is the red one
  bool okr[K], okb[K];            // interior
  int ro[K], rs[K], rn[K];        // the red cell's outside, south, north entries (black plane)
  int bo[K], bs[K], bn[K];        // the black cell's (red plane)
  float pr[K], pb[K], fr[K], fb[K];
  CellRule rr[K], rb[K];

  __device__ __forceinline__ void locate(const LdsLevel &L) {
#pragma unroll
    for (int k = 0; k < K; k++) {
      t[k] = (int)threadIdx.x + k * TPB_C;
      const int i = i0[k] = 2 * t[k];
      const int y = y0[k] = L.row_of(i), x = x0[k] = i - y * L.w;
      // a pair that wraps into the next row is two ring cells
      const bool row = i < L.n && y >= 1 && y <= L.h - 2;
      const bool ok0 = row && x >= 1 && x <= L.w - 2, ok1 = row && x + 1 <= L.w - 2;
      const bool rf = rfirst[k] = ((x + y) & 1) != 0;
      okr[k] = rf ? ok0 : ok1;
      okb[k] = rf ? ok1 : ok0;
      const int ir = rf ? i : i + 1, ib = rf ? i + 1 : i;
      ro[k] = (2 * ir - ib) >> 1;
      rs[k] = (ir - L.w) >> 1;
      rn[k] = (ir + L.w) >> 1;
      bo[k] = (2 * ib - ir) >> 1;
      bs[k] = (ib - L.w) >> 1;
      bn[k] = (ib + L.w) >> 1;
    }
  }
  // f and the rules of the interior cells, with the pair's two masks
  __device__ __forceinline__ void decode(const LdsLevel &L, int k, unsigned m0, unsigned m1) {
    const unsigned mr = rfirst[k] ? m0 : m1, mb = rfirst[k] ? m1 : m0;
    rr[k] = cell_rule(mr, rfirst[k], fr[k], L.hh);
    rb[k] = cell_rule(mb, !rfirst[k], fb[k], L.hh);
    // the first cell's outside neighbour lies west of the pair, the second's east
  }
  // f and the masks from LDS; ZERO: p is zero, else read
  template <bool ZERO> __device__ __forceinline__ void load(const LdsLevel &L) {
#pragma unroll
    for (int k = 0; k < K; k++) {
      const bool any = okr[k] || okb[k];
      fr[k] = any ? L.Fv[t[k]] : 0.0f;
      fb[k] = any ? L.Fv[L.half + t[k]] : 0.0f;
      const unsigned m = any ? *(const uint16_t *)(L.M + i0[k]) : 0u;
      pr[k] = !ZERO && any ? L.P[t[k]] : 0.0f;
      pb[k] = !ZERO && any ? L.P[L.half + t[k]] : 0.0f;
      decode(L, k, m & 0xffu, m >> 8);
    }
  }
  __device__ __forceinline__ void red(const LdsLevel &L, float alpha) {
    float *R = L.P, *B = L.P + L.half;
#pragma unroll
    for (int k = 0; k < K; k++)
      if (okr[k]) {
        pr[k] = smooth_rule(pr[k], B[ro[k]], pb[k], B[rs[k]], B[rn[k]], rr[k], alpha);
        R[t[k]] = pr[k];
      }
  }
  __device__ __forceinline__ void black(const LdsLevel &L, float alpha) {
    float *R = L.P, *B = L.P + L.half;
#pragma unroll
    for (int k = 0; k < K; k++)
      if (okb[k]) {
        pb[k] = smooth_rule(pb[k], R[bo[k]], pr[k], R[bs[k]], R[bn[k]], rb[k], alpha);
        B[t[k]] = pb[k];
      }
  }
  __device__ __forceinline__ void sweeps(const LdsLevel &L, int nu, float alpha, bool one_wave) {
    for (int s = 0; s < nu; s++) {
      red(L, alpha);
      phase_end(one_wave);
      black(L, alpha);
      phase_end(one_wave);
    }
  }
  // the interior cells' residuals into the planes at Q
  __device__ __forceinline__ void residual(const LdsLevel &L, float *Q) {
    const float *R = L.P, *B = L.P + L.half;
#pragma unroll
    for (int k = 0; k < K; k++) {
      if (okr[k])
        Q[t[k]] = residual_rule(pr[k], B[ro[k]], pb[k], B[rs[k]], B[rn[k]], fr[k], rr[k], L.ihsq);
      if (okb[k])
        Q[L.half + t[k]] =
            residual_rule(pb[k], R[bo[k]], pr[k], R[bs[k]], R[bn[k]], fb[k], rb[k], L.ihsq);
    }
  }
  // prolongate + correct (pressure_solver.cpp:134-181): a cell in an even row
  // takes coarse row y / 2, in an odd row also the one above, and likewise
  // the columns
  __device__ __forceinline__ void correct(const LdsLevel &L, const LdsLevel &C) {
    auto E = [&](int i, int x, int y) { return C.plane(C.P, !((x + y) & 1))[i >> 1]; };
#pragma unroll
    for (int k = 0; k < K; k++) {
      if (!(okr[k] || okb[k])) continue;
      // the pair holds an even column xe and an odd one xo: xo = xe + 1 or,
      // where an odd width shifts the pairs, xe - 1; coarse columns a, a + 1
      // under the odd one
      const bool efirst = !(x0[k] & 1);
      const int y = y0[k], xe = efirst ? x0[k] : x0[k] + 1, xo = efirst ? x0[k] + 1 : x0[k];
      const bool odd_row = (y & 1) != 0;
      const int by = y >> 1, ae = xe >> 1, ao = xo >> 1;
      const bool up = !odd_row || y <= L.h - 3; // an odd row needs the coarse row above
      const int by1 = odd_row && up ? by + 1 : by;
      const int ao1 = min(ao + 1, C.w - 1);
      const int c0 = by * C.w, c1 = by1 * C.w;
      // coarse values under the odd column (a, a + 1) x (b, b + 1); the even
      // column is a or a + 1
      const float e00 = E(c0 + ao, ao, by), e10 = E(c0 + ao1, ao1, by);
      const float e01 = E(c1 + ao, ao, by1), e11 = E(c1 + ao1, ao1, by1);
      const int f00 = C.M[c0 + ao] & MK_SELF, f10 = C.M[c0 + ao1] & MK_SELF;
      const int f01 = C.M[c1 + ao] & MK_SELF, f11 = C.M[c1 + ao1] & MK_SELF;
      const float g0 = ae == ao ? e00 : e10, g1 = ae == ao ? e01 : e11;
      const int q0 = ae == ao ? f00 : f10, q1 = ae == ao ? f01 : f11;
      const bool even_red = efirst == rfirst[k];
      const float Fe = even_red ? rr[k].F : rb[k].F, Fo = even_red ? rb[k].F : rr[k].F;
      const float ee = odd_row ? Fe * (g0 + g1) / eps_sum(q0 + q1) : g0 * Fe;
      const float num = odd_row ? e00 + e11 + e10 + e01 : e00 + e10;
      const float eo = Fo * num / eps_sum(odd_row ? f00 + f11 + f10 + f01 : f00 + f10);
      const float de = up ? ee : 0.0f, dn = up && xo <= L.w - 3 ? eo : 0.0f;
      if (okr[k]) L.P[t[k]] = pr[k] += even_red ? de : dn;
      if (okb[k]) L.P[L.half + t[k]] = pb[k] += even_red ? dn : de;
    }
  }
};

// restrict (pressure_solver.cpp:118-132) the residual planes Q of level L
// into the coarse level's f, a coarse cell per thread
__device__ __forceinline__ void lds_restrict(const LdsLevel &L, const LdsLevel &C, const float *Q) {
  const float *R = Q, *B = Q + L.half;
  for (int i = threadIdx.x; i < C.n; i += TPB_C) {
    const int Y = C.row_of(i), X = i - Y * C.w;
    if (Y < 1 || Y > C.h - 2 || X < 1 || X > C.w - 2) continue;
    const int j = (2 * Y) * L.w + 2 * X, js = j - L.w, jn = j + L.w;
    float v = 0.0f;
    v = B[(js - 1) >> 1] * 1.0f + R[js >> 1] * 2.0f + B[(js + 1) >> 1] * 1.0f;
    v += R[(j - 1) >> 1] * 2.0f + B[j >> 1] * 4.0f + R[(j + 1) >> 1] * 2.0f;
    v += B[(jn - 1) >> 1] * 1.0f + R[jn >> 1] * 2.0f + B[(jn + 1) >> 1] * 1.0f;
    C.plane(C.Fv, !((X + Y) & 1))[i >> 1] = v * (1.0f / 16.0f);
  }
}

// a wave that owns no pair of the level only meets its barriers
__device__ __forceinline__ bool idle_wave(const LdsLevel &L) {
  return __builtin_amdgcn_readfirstlane((int)threadIdx.x & ~63) >= L.half;
}

// the levels below the first one, whose residual the planes Q hold on entry:
// down to the coarsest and back up to the second, whose p is final on return
__device__ __forceinline__ void lds_inner(const CoarseArgs &a, char *smem, float *Q) {
  for (int l = 1; l < a.n; l++) {
    const LdsLevel L = lds_level(a, smem, l);
    lds_restrict(lds_level(a, smem, l - 1), L, Q);
    __syncthreads();
    const bool last = l == a.n - 1;
    const int nu = last ? a.nu_coarse : a.nu_pre;
    const bool one_wave = L.half <= 64;
    if (idle_wave(L)) {
      if (!one_wave)
        for (int s = 0; s < 2 * nu; s++) __syncthreads();
    } else {
      LevelPairs<1> t;
      t.locate(L);
      t.template load<true>(L);
      t.sweeps(L, nu, a.alpha, one_wave);
      if (!last) t.residual(L, Q);
    }
    __syncthreads();
  }
  for (int l = a.n - 2; l >= 1; l--) {
    const LdsLevel L = lds_level(a, smem, l), C = lds_level(a, smem, l + 1);
    const bool one_wave = L.half <= 64;
    if (idle_wave(L)) {
      if (!one_wave)
        for (int s = 0; s < 2 * a.nu_post + 1; s++) __syncthreads();
    } else {
      LevelPairs<1> t;
      t.locate(L);
      t.template load<false>(L);
      t.correct(L, C);
      phase_end(one_wave);
      t.sweeps(L, a.nu_post, a.alpha, one_wave);
    }
    __syncthreads();
  }
}

// p = 0 on every level and the masks of the levels below the first one in LDS.
// The masks' first TPB_C bytes of up to KR levels are loaded by load() in one
// round, which the caller issues along with its own loads.
struct CoarseInit {
  static constexpr int KR = 4;
  uint8_t rm[KR];
  __device__ __forceinline__ void load(const CoarseArgs &a) {
#pragma unroll
    for (int r = 0; r < KR; r++)
      if (1 + r < a.n && (int)threadIdx.x < a.w[1 + r] * a.h[1 + r])
        rm[r] = a.mask[1 + r][threadIdx.x];
  }
  __device__ __forceinline__ void store(const CoarseArgs &a, char *smem) const {
    const int tid = threadIdx.x;
    for (int l = 0; l < a.n; l++) {
      float *P = (float *)(smem + a.op[l]);
      const int m = (a.w[l] * a.h[l] + 1) & ~1;
      for (int i = tid; i < m; i += TPB_C) P[i] = 0.0f;
    }
#pragma unroll
    for (int r = 0; r < KR; r++)
      if (1 + r < a.n && tid < a.w[1 + r] * a.h[1 + r])
        ((uint8_t *)(smem + a.om[1 + r]))[tid] = rm[r];
    for (int l = 1; l < a.n; l++) {
      const int n = a.w[l] * a.h[l];
      for (int i = tid + (l <= KR ? TPB_C : 0); i < n; i += TPB_C)
        ((uint8_t *)(smem + a.om[l]))[i] = a.mask[l][i];
    }
  }
};

// the first level with K pairs per thread, in registers throughout.  ALONE: it
// is the coarsest one too
template <int K, bool ALONE>
__device__ __forceinline__ void lds_top(const CoarseArgs &a, char *smem, const float *f0,
                                        float *p0) {
  const LdsLevel L = lds_level(a, smem, 0);
  float *Q = (float *)(smem + a.orr);
  // every load before the first wait; a second cell past the level's end is
  // not there
  const uint8_t *m0 = a.mask[0];
  float fa[K], fb[K];
  unsigned ma[K], mb[K];
#pragma unroll
  for (int k = 0; k < K; k++) {
    const int i = 2 * ((int)threadIdx.x + k * TPB_C);
    const bool in0 = i < L.n, in1 = i + 1 < L.n;
    fa[k] = in0 ? f0[i] : 0.0f;
    fb[k] = in1 ? f0[i + 1] : 0.0f;
    ma[k] = in0 ? m0[i] : 0u;
    mb[k] = in1 ? m0[i + 1] : 0u;
  }
  CoarseInit init;
  init.load(a);
  LevelPairs<K> t;
  t.locate(L);
  init.store(a, smem);
#pragma unroll
  for (int k = 0; k < K; k++) {
    t.fr[k] = t.rfirst[k] ? fa[k] : fb[k];
    t.fb[k] = t.rfirst[k] ? fb[k] : fa[k];
    t.pr[k] = t.pb[k] = 0.0f;
    t.decode(L, k, ma[k], mb[k]);
  }
  __syncthreads();
  if (ALONE || a.n == 1) {
    t.sweeps(L, a.nu_coarse, a.alpha, false);
  } else {
    t.sweeps(L, a.nu_pre, a.alpha, false);
    t.residual(L, Q);
    __syncthreads();
    lds_inner(a, smem, Q);
    t.correct(L, lds_level(a, smem, 1));
    __syncthreads();
    t.sweeps(L, a.nu_post, a.alpha, false);
  }
#pragma unroll
  for (int k = 0; k < K; k++) {
    const float pa = t.rfirst[k] ? t.pr[k] : t.pb[k], pb = t.rfirst[k] ? t.pb[k] : t.pr[k];
    if (t.i0[k] < L.n) p0[t.i0[k]] = pa;
    if (t.i0[k] + 1 < L.n) p0[t.i0[k] + 1] = pb;
  }
}

// The whole V-cycle of levels first..L-2 of one domain in LDS, by one
// 1024-thread workgroup; f0 is the first level's rhs, the first level's
// solution is written to p0.  A first level of more than kCoarseMaxCells
// cells is taken only where no smaller one exists (very elongated domains),
// so it is the coarsest level too: BIG, a variant of its own because it needs
// more registers (all 128 that 1024 threads have, and five in scratch, against
// 118).
template <bool BIG>
__device__ __forceinline__ void coarse_vcycle_body(const CoarseArgs &a, const float *f0,
                                                  float *p0) {
  extern __shared__ __align__(16) char smem[];
  const int pairs = (a.w[0] * a.h[0] + 1) >> 1;
  if (pairs <= TPB_C) lds_top<1, false>(a, smem, f0, p0);
  else if (pairs <= 2 * TPB_C) lds_top<2, false>(a, smem, f0, p0);
  else if (BIG && pairs <= 4 * TPB_C) lds_top<4, true>(a, smem, f0, p0);
  else if (BIG) lds_top<6, true>(a, smem, f0, p0);
}
static_assert(kCoarseMaxCells == 4 * TPB_C && (size_t)2 * 6 * TPB_C * 13 >= LDS_BUDGET,
              "two pairs per thread; with BIG six, at 13 bytes of LDS a cell");
inline bool coarse_big(int w, int h) { return (size_t)w * h > kCoarseMaxCells; }

// LDS layout (p, f, mask per level, 16-byte aligned) of levels first..L-2
// for level sizes ws/hs; fills the offsets of `a` if given.  Returns the
// byte count, or SIZE_MAX if there are more than MAXL levels.
inline size_t coarse_lds_layout(const int *ws, const int *hs, int first, int levels,
                                CoarseArgs *a) {
  size_t off = 0;
  int k = 0;
  for (int l = first; l <= levels - 2; l++, k++) {
    if (k >= MAXL) return (size_t)-1;
    size_t n = (size_t)ws[l] * hs[l];
    if (a) {
      a->iw[k] = 1.0f / (float)ws[l];
      a->op[k] = (int)off;
      a->of[k] = (int)(off + ((n * 4 + 15) & ~size_t(15)));
      a->om[k] = (int)(off + 2 * ((n * 4 + 15) & ~size_t(15)));
    }
    off += 2 * ((n * 4 + 15) & ~size_t(15)) + ((n + 15) & ~size_t(15));
  }
  if (a) a->orr = (int)off;
  off += ((size_t)ws[first] * hs[first] * 4 + 15) & ~size_t(15);
  return off;
}

inline size_t coarse_lds_bytes(const Level *lv, int first, int levels, CoarseArgs *a) {
  int ws[64], hs[64];
  for (int l = 0; l < levels && l < 64; l++) {
    ws[l] = lv[l].w;
    hs[l] = lv[l].h;
  }
  return coarse_lds_layout(ws, hs, first, levels, a);
}

} // namespace ubg
