// mg_kernels.hip -- multigrid pressure-solver kernels for gfx950.
//
// Follows pressure_solver.cpp / pressure_solver.hpp of the reference:
//   smoothingKernel :10-24, rbgs :49-89 (two-pass red/black semantics),
//   calculateResidualField :91-116, restrict :118-132, prolongate :134-172,
//   correct :174-181, setZeroGradientBC :183-192, updateFields hpp:34-57.
// All kernels are memory-bound stencils (no MFMA); each thread owns one cell
// and one wave64 covers 64 consecutive cells of a row, so every load and store
// of a wave is one contiguous 256-byte segment.
#include "ubg_internal.hpp"

namespace ubg {

namespace {

constexpr int TPB = 256;

inline unsigned ceil_div(size_t a, size_t b) { return (unsigned)((a + b - 1) / b); }

__global__ void k_fill_f32(float *__restrict__ d, size_t n, float v) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) d[i] = v;
}
__global__ void k_fill_f64(double *__restrict__ d, size_t n, double v) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  size_t stride = (size_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) d[i] = v;
}
__global__ void k_f32_from_u8(const uint8_t *__restrict__ s, float *__restrict__ d, size_t n) {
  size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) d[i] = (float)s[i];
}

// Sum of squares, accumulated in double: block reduction through LDS, one
// atomic per block.
__global__ void k_sumsq(const float *__restrict__ s, size_t n, double *acc) {
  __shared__ double red[TPB];
  double v = 0.0;
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (size_t)gridDim.x * blockDim.x) {
    double x = s[i];
    v += x * x;
  }
  red[threadIdx.x] = v;
  __syncthreads();
  for (int o = TPB / 2; o > 0; o >>= 1) {
    if ((int)threadIdx.x < o) red[threadIdx.x] += red[threadIdx.x + o];
    __syncthreads();
  }
  if (threadIdx.x == 0) atomicAdd(acc, red[0]);
}

// mask = own flag (bit 0) + the four neighbours' flags (bits 1-4) + their
// count (bits 5-7); neighbours outside the grid count as 0.
__global__ void k_build_mask(const uint8_t *__restrict__ fl, uint8_t *__restrict__ m, int w,
                             int h) {
  int x = blockIdx.x * blockDim.x + threadIdx.x;
  int y = blockIdx.y;
  if (x >= w) return;
  size_t i = (size_t)y * w + x;
  uint8_t b = fl[i] ? MK_SELF : 0;
  if (x > 0 && fl[i - 1]) b |= MK_W;
  if (x < w - 1 && fl[i + 1]) b |= MK_E;
  if (y > 0 && fl[i - w]) b |= MK_S;
  if (y < h - 1 && fl[i + w]) b |= MK_N;
  unsigned cnt = ((b >> 1) & 1) + ((b >> 2) & 1) + ((b >> 3) & 1) + ((b >> 4) & 1);
  m[i] = (uint8_t)(b | (cnt << 5));
}

// Coarse flags and neighbour masks of a hierarchy (updateFields,
// pressure_solver.hpp:40-57).  pressure_solver.hpp:43-56: coarse flag is 1 iff
// sum(w * f)/16 > 0.2 over the full-weighting stencil; for 0/1 fine flags that
// is the integer rule weighted count >= 4.  The coarse boundary is 1
// (fill(1.0), :41).
//
// The flags of level l + 1 need those of level l, so a launch a level (and one
// more for its mask, and a fill of the coarse fields) leaves a hierarchy's
// set-up to launch latency: at 1025x1025 20 launches of 2 to 8 us.  Here a
// workgroup takes a 64x64 tile of a level with the halo that four coarsenings
// reach (15 cells before it, 8 behind), keeps the flags of its levels in
// LDS and writes the tile's masks and coarse flags; a level of at most
// kClassRest cells and all below it are one workgroup's, bound by its
// passes' latency.  1025x1025: 8.6 + 9.6 us for two launches instead of 55 us
// and 18 launch gaps; the allocation-free V-cycle on it 126 -> 91 us.  (With
// three coarsenings a launch, and so a tail from 128x128 cells instead of
// 64x64, 8.3 + 14.9.)
//
// Flags are bytes 0 / 1, so four cells' masks are one word: each neighbour's
// bit and its count (bits 5..7) come from one multiply-add, and no byte of a
// sum exceeds 159.
constexpr int CLT = 64;           // cells of a tile
constexpr int CLP0 = 88, CLH0 = CLT + 23; // first level's LDS rows (words of 4 cells from X0 - 16)
constexpr int CLR1 = CLT / 2 + 11, CLR2 = CLT / 4 + 5, CLR3 = CLT / 8 + 2;
constexpr int kClassThreads = 1024, kClassRest = 16384;
typedef uint32_t word_u __attribute__((aligned(1)));
struct ClassStage {
  const uint8_t *src;     // flags of the first level
  uint8_t *copy;          // first level's flags as 0 / 1 (null: not written)
  uint8_t *flag[5], *mask[4];
  float *zero[5][3];      // fields of the coarse levels to clear (null: none)
  int w[5], h[5];
  int n;                  // levels below the first: 0 .. 4
};
// masks of one cell or of four, from their flags and their neighbours'
__device__ __forceinline__ unsigned mask_bytes(unsigned c, unsigned w, unsigned e, unsigned s,
                                               unsigned n) {
  static_assert(MK_SELF == 1 && MK_W == 2 && MK_E == 4 && MK_S == 8 && MK_N == 16, "mask bits");
  return c + w * 34u + e * 36u + s * 40u + n * 48u;
}
// coarse flag from the 3x3 fine flags around f (rows of `pitch` bytes)
__device__ __forceinline__ unsigned coarse_flag(const uint8_t *f, int pitch) {
  const uint8_t *r0 = f - pitch, *r2 = f + pitch;
  const int v = (r0[-1] + 2 * r0[0] + r0[1]) + 2 * (f[-1] + 2 * f[0] + f[1]) +
                (r2[-1] + 2 * r2[0] + r2[1]);
  return v >= 4 ? 1u : 0u;
}

__global__ void __launch_bounds__(kClassThreads) k_classify(ClassStage a) {
  constexpr int PW = CLP0 / 4;
  __shared__ uint32_t f0_[CLH0 * PW + 2];
  uint32_t *const f0 = f0_ + 1; // cell (x, y): byte x - X0 + 16 of row y - Y0 + 15
  __shared__ uint8_t f1[CLR1 * CLR1], f2[CLR2 * CLR2], f3[CLR3 * CLR3];
  const int X0 = blockIdx.x * CLT, Y0 = blockIdx.y * CLT, w0 = a.w[0], h0 = a.h[0];
  constexpr int NLD = (CLH0 * PW + kClassThreads - 1) / kClassThreads;
  uint32_t v0[NLD];
#pragma unroll
  for (int k = 0; k < NLD; k++) {
    const int i = threadIdx.x + k * kClassThreads;
    const int x = X0 - 16 + 4 * (i % PW), y = Y0 - 15 + i / PW;
    v0[k] = 0u;
    if (y < 0 || y >= h0 || i >= CLH0 * PW) continue;
    const uint8_t *row = a.src + (size_t)y * w0;
    if (x >= 0 && x + 4 <= w0) v0[k] = *(const word_u *)(row + x);
    else
      for (int c = 0; c < 4; c++)
        if (x + c >= 0 && x + c < w0) v0[k] |= (uint32_t)row[x + c] << (8 * c);
  }
#pragma unroll
  for (int k = 0; k < NLD; k++) {
    const int i = threadIdx.x + k * kClassThreads;
    uint32_t t = v0[k]; // bit 0 of a byte: the or of its bits
    t |= t >> 4;
    t |= t >> 2;
    t |= t >> 1;
    if (i < CLH0 * PW) f0[i] = t & 0x01010101u;
  }
  __syncthreads();
  { // the tile's masks, four cells a thread: 16 words x 64 rows
    static_assert(CLT / 4 * CLT == kClassThreads, "one word a thread");
    const int i = threadIdx.x % (CLT / 4), y = threadIdx.x / (CLT / 4), x = X0 + 4 * i;
    const uint32_t *r = f0 + (y + 15) * PW + i + 4;
    const uint32_t c = r[0], wst = (c << 8) | (r[-1] >> 24), e = (c >> 8) | (r[1] << 24);
    const uint32_t m = mask_bytes(c, wst, e, r[-PW], r[PW]);
    if (Y0 + y < h0) {
      const size_t o = (size_t)(Y0 + y) * w0 + x;
      if (x + 4 <= w0) {
        *(word_u *)(a.mask[0] + o) = m;
        if (a.copy) *(word_u *)(a.copy + o) = c;
      } else
        for (int k = 0; k < 4; k++)
          if (x + k < w0) {
            a.mask[0][o + k] = (uint8_t)(m >> (8 * k));
            if (a.copy) a.copy[o + k] = (uint8_t)(c >> (8 * k));
          }
    }
  }
  // cell (x, y) of the stage's level k with flag v, in LDS region r x r from
  // (x0, y0); the tile owns t x t cells from (x0 + lo, y0 + lo)
  auto put = [&](int k, int x, int y, unsigned v, uint8_t *out, int r, int lo, int t) {
    const int rx = x - ((X0 >> k) - lo), ry = y - ((Y0 >> k) - lo), w = a.w[k], h = a.h[k];
    if (rx < 0 || rx >= r || ry < 0 || ry >= r) return;
    const bool in = x >= 0 && x < w && y >= 0 && y < h;
    if (!in) v = 0;
    else if (x == 0 || x == w - 1 || y == 0 || y == h - 1) v = 1;
    if (out) out[ry * r + rx] = (uint8_t)v;
    if (in && rx >= lo && rx < lo + t && ry >= lo && ry < lo + t) {
      const size_t o = (size_t)y * w + x;
      a.flag[k][o] = (uint8_t)v;
      if (a.zero[k][0]) a.zero[k][0][o] = a.zero[k][1][o] = a.zero[k][2][o] = 0.0f;
    }
  };
  auto masks = [&](int k, const uint8_t *f, int r, int lo, int t) {
    for (int i = threadIdx.x; i < t * t; i += kClassThreads) {
      const int x = i % t, y = i / t, gx = (X0 >> k) + x, gy = (Y0 >> k) + y;
      if (gx >= a.w[k] || gy >= a.h[k]) continue;
      const uint8_t *q = f + (y + lo) * r + x + lo;
      a.mask[k][(size_t)gy * a.w[k] + gx] =
          (uint8_t)mask_bytes(q[0], q[-1], q[1], q[-r], q[r]);
    }
  };
  if (a.n < 1) return;
  // level 1, two cells of a row from a word: the column sums of its three
  // rows, then each byte with its neighbours (at most 16).  The first cell of
  // word 0 lies outside the region.
  static_assert(CLR1 * PW <= kClassThreads, "one word a thread");
  if (threadIdx.x < CLR1 * PW) {
    const int i = threadIdx.x % PW, ry = threadIdx.x / PW;
    const int y = (Y0 >> 1) - 7 + ry, x = (X0 - 16 + 4 * i) >> 1; // cells x, x + 1
    const uint32_t *r = f0 + (2 * ry + 1) * PW + i;               // row 2 y
    auto column = [&](int d) { return r[d - PW] + 2u * r[d] + r[d + PW]; };
    const uint32_t c = column(0), l = (c << 8) | (column(-1) >> 24);
    const uint32_t t = l + 2u * c + (c >> 8); // bytes 0 and 2 are whole
    put(1, x, y, (t & 0xffu) >= 4u, f1, CLR1, 7, CLT / 2);
    put(1, x + 1, y, ((t >> 16) & 0xffu) >= 4u, f1, CLR1, 7, CLT / 2);
  }
  __syncthreads();
  masks(1, f1, CLR1, 7, CLT / 2);
  // levels 2 .. 4: a region begins one cell into the double of the next
  auto coarsen = [&](int k, const uint8_t *fine, int fr, uint8_t *out, int r, int lo, int t) {
    if (threadIdx.x >= (unsigned)(r * r)) return;
    const int rx = threadIdx.x % r, ry = threadIdx.x / r;
    put(k, (X0 >> k) - lo + rx, (Y0 >> k) - lo + ry,
        coarse_flag(fine + (2 * ry + 1) * fr + 2 * rx + 1, fr), out, r, lo, t);
  };
  if (a.n < 2) return;
  coarsen(2, f1, CLR1, f2, CLR2, 3, CLT / 4);
  __syncthreads();
  masks(2, f2, CLR2, 3, CLT / 4);
  if (a.n < 3) return;
  coarsen(3, f2, CLR2, f3, CLR3, 1, CLT / 8);
  __syncthreads();
  masks(3, f3, CLR3, 1, CLT / 8);
  if (a.n < 4) return;
  coarsen(4, f3, CLR3, nullptr, CLT / 16, 0, CLT / 16);
}

// the level of at most kClassRest cells and all below it: level k's flags in
// one LDS buffer, level k + 1's into the other, each with a ring of zeros
struct ClassRest {
  const uint8_t *src;
  uint8_t *copy;
  uint8_t *flag[16], *mask[16];
  float *zero[16][3];
  int w[16], h[16];
  int n; // levels below the first
};
constexpr int kClassRing = kClassRest + 2 * (kClassRest / 4 + 4) + 4; // (w + 2)(h + 2), w, h >= 4
__global__ void __launch_bounds__(1024) k_classify_rest(ClassRest a) {
  __shared__ uint8_t buf[2][kClassRing];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // rings: the cells of a level are written between the barriers
  auto ring = [&](uint8_t *f, int w, int h) {
    for (int i = threadIdx.x; i < w + 2; i += 1024) f[i] = f[(h + 1) * (w + 2) + i] = 0;
    for (int i = threadIdx.x; i < h; i += 1024) f[(i + 1) * (w + 2)] = f[(i + 2) * (w + 2) - 1] = 0;
  };
  const int w0 = a.w[0], h0 = a.h[0];
  ring(buf[0], w0, h0);
  for (int x = lane; x < w0; x += 64)
    for (int y = wave; y < h0; y += 16 * 8) { // eight loads in flight
      uint8_t v[8];
#pragma unroll
      for (int j = 0; j < 8; j++) v[j] = a.src[min(y + 16 * j, h0 - 1) * w0 + x];
#pragma unroll
      for (int j = 0; j < 8; j++) {
        if (y + 16 * j >= h0) break;
        v[j] = v[j] != 0 ? 1 : 0;
        buf[0][(y + 16 * j + 1) * (w0 + 2) + x + 1] = v[j];
        if (a.copy) a.copy[(y + 16 * j) * w0 + x] = v[j];
      }
    }
  __syncthreads();
  for (int k = 0;; k++) {
    const int w = a.w[k], h = a.h[k], p = w + 2;
    const uint8_t *f = buf[k & 1] + p + 1; // cell (0, 0)
    uint8_t *const mask = a.mask[k];
    for (int x = lane; x < w; x += 64)
#pragma unroll 4
      for (int y = wave; y < h; y += 16) {
        const uint8_t *q = f + y * p + x;
        mask[y * w + x] = (uint8_t)mask_bytes(q[0], q[-1], q[1], q[-p], q[p]);
      }
    if (k == a.n) return;
    const int wc = a.w[k + 1], hc = a.h[k + 1];
    uint8_t *c = buf[(k + 1) & 1];
    ring(c, wc, hc);
    c += wc + 3;
    uint8_t *const flag = a.flag[k + 1];
    float *const z0 = a.zero[k + 1][0], *const z1 = a.zero[k + 1][1], *const z2 = a.zero[k + 1][2];
    for (int x = lane; x < wc; x += 64)
#pragma unroll 2
      for (int y = wave; y < hc; y += 16) {
        const int i = y * wc + x;
        const unsigned v = x == 0 || x == wc - 1 || y == 0 || y == hc - 1
                               ? 1u
                               : coarse_flag(f + 2 * y * p + 2 * x, p);
        c[y * (wc + 2) + x] = (uint8_t)v;
        flag[i] = (uint8_t)v;
        if (z0) z0[i] = z1[i] = z2[i] = 0.0f;
      }
    __syncthreads();
  }
}

// setZeroGradientBC (pressure_solver.cpp:183-192): edges copy the first
// interior cell; corners untouched.  No read depends on another write.
__global__ void k_zero_gradient(float *__restrict__ p, int w, int h) {
  int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= 1 && t < h - 1) {
    size_t r = (size_t)t * w;
    p[r] = p[r + 1];
    p[r + w - 1] = p[r + w - 2];
  }
  if (t >= 1 && t < w - 1) {
    p[t] = p[(size_t)w + t];
    p[(size_t)(h - 1) * w + t] = p[(size_t)(h - 2) * w + t];
  }
}

// calculateResidualField for one interior cell (pressure_solver.cpp:100-108):
// r = F*(f + (sum_n(F_n p_n + (1-F_n) p) - 4p) / h^2), neighbours summed in
// the order x-1, x+1, y-1, y+1.
__device__ __forceinline__ float residual_cell(const float *__restrict__ p,
                                               const float *__restrict__ f,
                                               const uint8_t *__restrict__ m, size_t i, int w,
                                               float ihsq) {
  uint8_t mk = m[i];
  float pc = p[i];
  float val = 0.0f;
  val += (mk & MK_W) ? p[i - 1] : pc;
  val += (mk & MK_E) ? p[i + 1] : pc;
  val += (mk & MK_S) ? p[i - w] : pc;
  val += (mk & MK_N) ? p[i + w] : pc;
  val += -4.0f * pc;
  val *= ihsq;
  return (mk & MK_SELF) ? (f[i] + val) : 0.0f;
}

__global__ void k_residual(const float *__restrict__ p, const float *__restrict__ f,
                           const uint8_t *__restrict__ m, float *__restrict__ r, int w,
                           float ihsq) {
  int x = blockIdx.x * blockDim.x + threadIdx.x + 1;
  int y = blockIdx.y + 1;
  if (x >= w - 1) return;
  size_t i = (size_t)y * w + x;
  r[i] = residual_cell(p, f, m, i, w, ihsq);
}

// Fused calculateResidualField + restrict (pressure_solver.cpp:217-227): the
// fine residual never reaches HBM.  Each thread owns one coarse interior cell,
// computes the nine fine residuals under the full-weighting stencil and
// writes the coarse right-hand side; the coarse solution starts at zero
// (ec.fill(0.0), :224).
__global__ void k_residual_restrict(const float *__restrict__ p, const float *__restrict__ f,
                                    const uint8_t *__restrict__ m, int wf, float ihsq,
                                    float *__restrict__ rc, float *__restrict__ ec, int wc) {
  int x = blockIdx.x * blockDim.x + threadIdx.x + 1;
  int y = blockIdx.y + 1;
  if (x >= wc - 1) return;
  size_t c = (size_t)(2 * y) * wf + 2 * x;
  auto R = [&](int dx, int dy) { return residual_cell(p, f, m, c + (ptrdiff_t)dy * wf + dx, wf, ihsq); };
  float v = 0.0f;
  v = R(-1, -1) * 1.0f + R(0, -1) * 2.0f + R(1, -1) * 1.0f;
  v += R(-1, 0) * 2.0f + R(0, 0) * 4.0f + R(1, 0) * 2.0f;
  v += R(-1, 1) * 1.0f + R(0, 1) * 2.0f + R(1, 1) * 1.0f;
  size_t ci = (size_t)y * wc + x;
  rc[ci] = v * (1.0f / 16.0f);
  ec[ci] = 0.0f;
}

// LDS-tiled variant for large levels: a workgroup owns 32x8 coarse cells,
// computes the 65x17 fine residuals under them once into LDS (p staged with
// a one-cell halo, all loads issued before the first LDS store), then
// restricts.  Same arithmetic as k_residual_restrict.
constexpr int RCX = 32, RCY = 8;
constexpr int RFX = 2 * RCX + 1, RFY = 2 * RCY + 1;  // residual region
constexpr int RPX = RFX + 2, RPY = RFY + 2;          // p region
__global__ void __launch_bounds__(256)
    k_residual_restrict_tile(const float *__restrict__ p, const float *__restrict__ f,
                             const uint8_t *__restrict__ m, int wf, int hf, float ihsq,
                             float *__restrict__ rc, float *__restrict__ ec, int wc, int hc,
                             int ntx) {
  __shared__ float sp[RPY][RPX];
  __shared__ float sr[RFY][RFX + 1];
  const int tid = threadIdx.x;
  const int X0 = 1 + (blockIdx.x % ntx) * RCX, Y0 = 1 + (blockIdx.x / ntx) * RCY;
  const int fx0 = 2 * X0 - 1, fy0 = 2 * Y0 - 1; // residual region origin
  constexpr int NP = RPX * RPY, NPI = (NP + 255) / 256;
  float v[NPI];
#pragma unroll
  for (int k = 0; k < NPI; k++) {
    int li = tid + 256 * k;
    int r = li / RPX, c = li - r * RPX;
    int gx = fx0 - 1 + c, gy = fy0 - 1 + r;
    v[k] = (li < NP && gx >= 0 && gx < wf && gy >= 0 && gy < hf) ? p[(size_t)gy * wf + gx] : 0.0f;
  }
#pragma unroll
  for (int k = 0; k < NPI; k++) {
    int li = tid + 256 * k;
    if (li < NP) (&sp[0][0])[li] = v[k];
  }
  __syncthreads();
  for (int li = tid; li < RFX * RFY; li += 256) {
    int r = li / RFX, c = li - r * RFX;
    int gx = fx0 + c, gy = fy0 + r;
    float res = 0.0f;
    if (gx >= 1 && gx < wf - 1 && gy >= 1 && gy < hf - 1) {
      size_t gi = (size_t)gy * wf + gx;
      unsigned mk = m[gi];
      float pc = sp[r + 1][c + 1];
      float val = 0.0f;
      val += (mk & MK_W) ? sp[r + 1][c] : pc;
      val += (mk & MK_E) ? sp[r + 1][c + 2] : pc;
      val += (mk & MK_S) ? sp[r][c + 1] : pc;
      val += (mk & MK_N) ? sp[r + 2][c + 1] : pc;
      val += -4.0f * pc;
      val *= ihsq;
      res = (mk & MK_SELF) ? (f[gi] + val) : 0.0f;
    }
    sr[r][c] = res;
  }
  __syncthreads();
  const int cx = tid % RCX, cy = tid / RCX; // 256 threads = 32 x 8 coarse cells
  const int X = X0 + cx, Y = Y0 + cy;
  if (X < wc - 1 && Y < hc - 1) {
    const int r = 2 * cy + 1, c = 2 * cx + 1; // fine (2X, 2Y) in the residual region
    auto R = [&](int dx, int dy) { return sr[r + dy][c + dx]; };
    float vv = 0.0f;
    vv = R(-1, -1) * 1.0f + R(0, -1) * 2.0f + R(1, -1) * 1.0f;
    vv += R(-1, 0) * 2.0f + R(0, 0) * 4.0f + R(1, 0) * 2.0f;
    vv += R(-1, 1) * 1.0f + R(0, 1) * 2.0f + R(1, 1) * 1.0f;
    size_t ci = (size_t)Y * wc + X;
    rc[ci] = vv * (1.0f / 16.0f);
    ec[ci] = 0.0f;
  }
}

// flag sum + the double literal 0.0001, stored as float (pressure_solver.cpp:149)
__device__ __forceinline__ float eps_sum(int s) { return (float)((double)s + 0.0001); }

// Fused prolongate + correct (pressure_solver.cpp:134-181): e is computed per
// fine interior cell by its parity class and added to p; cells the
// reference's loops do not reach (last odd column/row of an odd-sized grid)
// keep e = 0.
__global__ void k_prolong_correct(float *__restrict__ p, const uint8_t *__restrict__ m, int w,
                                  int h, const float *__restrict__ ec,
                                  const uint8_t *__restrict__ fc, int wc) {
  int x = blockIdx.x * blockDim.x + threadIdx.x + 1;
  int y = blockIdx.y + 1;
  if (x >= w - 1) return;
  size_t i = (size_t)y * w + x;
  float F = (m[i] & MK_SELF) ? 1.0f : 0.0f;
  int a = x >> 1, b = y >> 1;
  bool xe = !(x & 1), ye = !(y & 1);
  auto E = [&](int xx, int yy) { return ec[(size_t)yy * wc + xx]; };
  auto FC = [&](int xx, int yy) { return (int)fc[(size_t)yy * wc + xx]; };
  float e = 0.0f;
  if (xe && ye) {
    e = E(a, b) * F;
  } else if (!xe && ye) {
    if (x <= w - 3) e = F * (E(a, b) + E(a + 1, b)) / eps_sum(FC(a, b) + FC(a + 1, b));
  } else if (xe && !ye) {
    if (y <= h - 3) e = F * (E(a, b) + E(a, b + 1)) / eps_sum(FC(a, b) + FC(a, b + 1));
  } else {
    if (x <= w - 3 && y <= h - 3)
      e = F * (E(a, b) + E(a + 1, b + 1) + E(a + 1, b) + E(a, b + 1)) /
          eps_sum(FC(a, b) + FC(a + 1, b + 1) + FC(a + 1, b) + FC(a, b + 1));
  }
  p[i] += e;
}

} // namespace

// ---------------------------------------------------------------------------
void launch_fill_f32(float *dst, size_t n, float v, hipStream_t s) {
  if (!n) return;
  unsigned g = ceil_div(n, TPB);
  if (g > 4096) g = 4096;
  hipLaunchKernelGGL(k_fill_f32, dim3(g), dim3(TPB), 0, s, dst, n, v);
}
void launch_fill_f64(double *dst, size_t n, double v, hipStream_t s) {
  if (!n) return;
  unsigned g = ceil_div(n, TPB);
  if (g > 4096) g = 4096;
  hipLaunchKernelGGL(k_fill_f64, dim3(g), dim3(TPB), 0, s, dst, n, v);
}
void launch_f32_from_u8(const uint8_t *src, float *dst, size_t n, hipStream_t s) {
  if (!n) return;
  hipLaunchKernelGGL(k_f32_from_u8, dim3(ceil_div(n, TPB)), dim3(TPB), 0, s, src, dst, n);
}
void launch_sumsq(const float *src, size_t n, double *acc, hipStream_t s) {
  if (!n) return;
  unsigned g = ceil_div(n, TPB);
  if (g > 2048) g = 2048;
  hipLaunchKernelGGL(k_sumsq, dim3(g), dim3(TPB), 0, s, src, n, acc);
}
void launch_build_mask(const uint8_t *flag, uint8_t *mask, int w, int h, hipStream_t s) {
  hipLaunchKernelGGL(k_build_mask, dim3(ceil_div(w, TPB), h), dim3(TPB), 0, s, flag, mask, w, h);
}
void launch_classify(const Level *lv, int levels, const uint8_t *raw, bool zero, hipStream_t s) {
  int l = 0;
  const uint8_t *src = raw ? raw : lv[0].flag;
  uint8_t *copy = raw ? lv[0].flag : nullptr;
  for (; (size_t)lv[l].w * lv[l].h > kClassRest; l += 4) {
    ClassStage a{};
    a.src = src;
    a.copy = copy;
    a.n = levels - 1 - l < 4 ? levels - 1 - l : 4;
    for (int k = 0; k <= a.n; k++) {
      const Level &L = lv[l + k];
      a.w[k] = L.w;
      a.h[k] = L.h;
      a.flag[k] = L.flag;
      if (k < 4) a.mask[k] = L.mask;
      if (zero && k > 0) {
        a.zero[k][0] = L.p;
        a.zero[k][1] = L.p_alt;
        a.zero[k][2] = L.f;
      }
    }
    hipLaunchKernelGGL(k_classify, dim3(ceil_div(lv[l].w, CLT), ceil_div(lv[l].h, CLT)),
                       dim3(kClassThreads), 0, s, a);
    if (l + 4 > levels - 1) return; // the last level's mask is written
    src = lv[l + 4].flag;
    copy = nullptr;
  }
  ClassRest a{};
  a.src = src;
  a.copy = copy;
  a.n = levels - 1 - l;
  for (int k = 0; k <= a.n; k++) {
    const Level &L = lv[l + k];
    a.w[k] = L.w;
    a.h[k] = L.h;
    a.flag[k] = L.flag;
    a.mask[k] = L.mask;
    if (zero && k > 0) {
      a.zero[k][0] = L.p;
      a.zero[k][1] = L.p_alt;
      a.zero[k][2] = L.f;
    }
  }
  hipLaunchKernelGGL(k_classify_rest, dim3(1), dim3(1024), 0, s, a);
}
void launch_zero_gradient(float *p, int w, int h, hipStream_t s) {
  int n = w > h ? w : h;
  hipLaunchKernelGGL(k_zero_gradient, dim3(ceil_div(n, TPB)), dim3(TPB), 0, s, p, w, h);
}
void launch_residual(const Level &L, float h, hipStream_t s) {
  float ihsq = 1.0f / h / h;
  hipLaunchKernelGGL(k_residual, dim3(ceil_div(L.w - 2, TPB), L.h - 2), dim3(TPB), 0, s, L.p,
                     L.f, L.mask, L.r, L.w, ihsq);
}
void launch_residual_restrict(const Level &F, const Level &C, float h, hipStream_t s) {
  if (C.w < 3 || C.h < 3) return;
  float ihsq = 1.0f / h / h;
  if ((size_t)C.w * C.h >= 16384) {
    int ntx = (C.w - 2 + RCX - 1) / RCX, nty = (C.h - 2 + RCY - 1) / RCY;
    hipLaunchKernelGGL(k_residual_restrict_tile, dim3(ntx * nty), dim3(256), 0, s, F.p, F.f,
                       F.mask, F.w, F.h, ihsq, C.f, C.p, C.w, C.h, ntx);
  } else {
    hipLaunchKernelGGL(k_residual_restrict, dim3(ceil_div(C.w - 2, TPB), C.h - 2), dim3(TPB), 0,
                       s, F.p, F.f, F.mask, F.w, ihsq, C.f, C.p, C.w);
  }
}
void launch_prolong_correct(const Level &F, const Level &C, hipStream_t s) {
  hipLaunchKernelGGL(k_prolong_correct, dim3(ceil_div(F.w - 2, TPB), F.h - 2), dim3(TPB), 0, s,
                     F.p, F.mask, F.w, F.h, C.p, C.flag, C.w);
}

} // namespace ubg
