// regtile_device.hpp -- multigrid level passes (MG::solveLevel,
// pressure_solver.cpp:201-248) with the tile held in registers, as device
// functions over one tile:
//   pre : NU red/black sweeps, residual, full-weighting restriction
//   post: prolongation, correction, NU red/black sweeps
// with setZeroGradientBC (:183-192) after every sweep and after the
// correction where the level takes it (ZG).
//
// Layout.  A workgroup of WAVES waves covers a region of 128 columns and
// WAVES RPW rows: lane l of wave v holds columns gx0 + 2l + c (c < 2) of
// rows gy0 + RPW v + i (i < RPW) -- p, f and the mask bytes of 2 RPW cells.
// gx0 and gy0 are even, so the colour (x + y) & 1 of a register is (c + i) & 1
// whatever the lane.  Of a cell's four neighbours most sit in the same lane;
// the ones left and right of the lane come by a DPP lane shift, and a wave
// publishes its first and last row through LDS after each colour phase
// (`below` / `above` hold the neighbouring waves' rows).  So a phase costs
// one barrier and two half-row exchanges per wave instead of six LDS
// accesses per cell, and f and the mask are read once.
//
// Halo.  A value is exact if it lies as many cells inside the region as
// colour phases have run, so the region carries 2 cells per sweep around the
// owned otx x oty cells (plus the reach of the residual and the restriction);
// halo cells are recomputed by the neighbouring tile from the same inputs.
// The sweeps read p and write p_out, so no tile sees another's new values and
// every owned cell is the value the sweep-by-sweep schedule produces, bit for
// bit.
//
// Uniform rows.  Where every interior cell of a wave's row has itself and its
// four neighbours fluid (mask 0x9f) and alpha is 1, the update is
// (((0 + W) + E + S) + N + (f h) h) / 4: no selects, and a product with 0.25,
// which rounds as the division does.  One ballot per row decides it for all
// sweeps; other rows take the constants from the LDS rule table.  A sum that
// overflows gives NaN in both (the rule's quotient is corrected by v - 4 q =
// inf - inf), so that a cell's value does not depend on the row and tile that
// compute it.
#pragma once

#include "mg_device.hpp"

namespace ubg {

// The smoothing constants of every mask byte, for passes that look them up
// in LDS instead of decoding the byte at each update: entry 2 mk holds the
// four neighbour selectors (0 / -1 for the bits W, E, S, N), entry 2 mk + 1
// RN(1/s) and -s for the neighbour count s, the quotient's select (0 when
// s == 0, else -1) and F, as bits.  Filled by the whole workgroup.
constexpr int kRuleEntries = 512;
__device__ __forceinline__ void fill_rule_table(uint4 *tab) {
  for (unsigned mk = threadIdx.x; mk < 256u; mk += blockDim.x) {
    const unsigned s = mk >> 5;
    const float pow2 = __int_as_float((int)((127u - (s >> 1)) << 23));
    const float inv = (s == 3u) ? (1.0f / 3.0f) : pow2;
    tab[2 * mk] = make_uint4(0u - ((mk >> 1) & 1u), 0u - ((mk >> 2) & 1u), 0u - ((mk >> 3) & 1u),
                             0u - ((mk >> 4) & 1u));
    tab[2 * mk + 1] = make_uint4(__float_as_uint(inv), __float_as_uint(-(float)s),
                                 s == 0u ? 0u : ~0u, __float_as_uint((float)(mk & MK_SELF)));
  }
}
// smooth_fhh with the mask's constants from the table: the same operations
// in the same order (keep_if, div_count, the zero-count case, F), so the
// same value.
__device__ __forceinline__ float smooth_tab(float pc, float pw, float pe, float ps, float pn,
                                            float fhh, const uint4 *tab, unsigned mk,
                                            float alpha) {
  const uint4 nb = tab[2 * mk], dc = tab[2 * mk + 1];
  float val = 0.0f;
  val += __uint_as_float(__float_as_uint(pw) & nb.x);
  val += __uint_as_float(__float_as_uint(pe) & nb.y);
  val += __uint_as_float(__float_as_uint(ps) & nb.z);
  val += __uint_as_float(__float_as_uint(pn) & nb.w);
  val += fhh;
  const float inv = __uint_as_float(dc.x);
  const float q = val * inv;
  const float r = fmaf(__uint_as_float(dc.y), q, val);
  const float q2 = fmaf(r, inv, q);
  val = __uint_as_float(__float_as_uint(q2) & dc.z);
  return __uint_as_float(dc.w) * (alpha * val + (1.0f - alpha) * pc);
}

// a lane's two cells at element alignment: a row starts at any multiple of 4
// bytes, and gfx950 loads and stores a dword pair at any such address
typedef float pair_u __attribute__((ext_vector_type(2), aligned(4)));
typedef uint16_t mpair_u __attribute__((aligned(1)));

// the value of the lane to the left / right (+0 beyond the wave's ends, which
// are halo cells): a DPP operand of the instruction that uses it
__device__ __forceinline__ float lane_left(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x138, 0xf, 0xf, true));
}
__device__ __forceinline__ float lane_right(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x130, 0xf, 0xf, true));
}
// keeps a uniform branch a branch (the compiler would turn the rare rows'
// code into selects that every wave executes)
__device__ __forceinline__ void stay_branch() { asm volatile(""); }

template <int NU_, int RPW_, int WAVES_> struct RegTile {
  static constexpr int NU = NU_, CPL = 2, RPW = RPW_, WAVES = WAVES_;
  static constexpr int TPB = 64 * WAVES, COLS = 64 * CPL, ROWS = RPW * WAVES;
  // waves per SIMD to compile the single-domain passes for: with 6 rows, three
  // workgroups of 8 waves or two of 12 a CU need 6 (82 registers instead of 80
  // leave one less: pre without the zero-gradient BC 39.9 instead of 34.5 us at
  // 4096x2048, 189 instead of 129 with 12 waves at 8192x4096).  Without the
  // zero-gradient BC pre reaches 80 (at two and three sweeps) by keeping two of
  // them in scratch, 12 bytes a lane, which those times include; with it pre
  // needs 79, post 66.  The batched passes, which also walk their
  // tiles, spill more under that bound (24.9 us instead of 22.9) and keep 4.
  static constexpr int MINW = RPW >= 6 ? 6 : 4;
  static_assert(RPW % 2 == 0, "a register's colour does not depend on the wave");
  // pre: residuals on [X0-1, X0+otx-1] read p on [X0-2, X0+otx]; each sweep
  // widens that by 2
  static constexpr int HXP = 2 + 2 * NU, HYP = 2 + 2 * NU;
  static constexpr int OTXP = (COLS - HXP - (2 * NU + 1)) / 2 * 2;
  static constexpr int OTYP = (ROWS - HYP - (2 * NU + 1)) / 2 * 2;
  // post: one more column on the right, whose correction lacks the lane
  // beyond the last
  static constexpr int HXQ = 2 * NU, HYQ = 2 * NU;
  static constexpr int OTXQ = (COLS - HXQ - (2 * NU + 1)) / 2 * 2;
  static constexpr int OTYQ = (ROWS - HYQ - 2 * NU) / 2 * 2;
  // LDS: rule table, three exchange buffers of two half rows per wave
  static constexpr int XROW = 64;               // floats
  static constexpr int XBUF = WAVES * 2 * XROW;
  // HOLD: the smoothing constants of the lane's cells are decoded once into
  // registers; else rows that are not uniform look them up in LDS per update
  static constexpr bool HOLD = RPW <= 2;
  static constexpr size_t TAB = HOLD ? 0 : sizeof(uint4) * kRuleEntries;
  static constexpr size_t LDS = TAB + 3 * XBUF * sizeof(float);
};

// a cell's smoothing constants as smooth_tab's table holds them
struct HeldRule {
  unsigned w, e, s, n, some; // selectors
  float inv, ns, F;
};
__device__ __forceinline__ HeldRule held_rule(unsigned mk) {
  HeldRule r;
  r.w = 0u - ((mk >> 1) & 1u);
  r.e = 0u - ((mk >> 2) & 1u);
  r.s = 0u - ((mk >> 3) & 1u);
  r.n = 0u - ((mk >> 4) & 1u);
  const unsigned c = mk >> 5;
  r.inv = c == 3u ? (1.0f / 3.0f) : __int_as_float((int)((127u - (c >> 1)) << 23));
  r.ns = -(float)c;
  r.some = c == 0u ? 0u : ~0u;
  r.F = (float)(mk & MK_SELF);
  return r;
}
__device__ __forceinline__ float smooth_held(float pc, float pw, float pe, float ps, float pn,
                                             float fhh, const HeldRule &r, float alpha) {
  float val = 0.0f;
  val += __uint_as_float(__float_as_uint(pw) & r.w);
  val += __uint_as_float(__float_as_uint(pe) & r.e);
  val += __uint_as_float(__float_as_uint(ps) & r.s);
  val += __uint_as_float(__float_as_uint(pn) & r.n);
  val += fhh;
  const float q = val * r.inv;
  const float q2 = fmaf(fmaf(r.ns, q, val), r.inv, q);
  val = __uint_as_float(__float_as_uint(q2) & r.some);
  return r.F * (alpha * val + (1.0f - alpha) * pc);
}

// The shapes in use, and which a pass takes by the number of tiles its level
// splits into (the batched solver: its members' tiles together).  Up to one
// workgroup per CU a launch is all latency, and the shape with the fewest
// waves whose tiles still fit is the fastest: 12 waves of 2 rows, then 16
// (256x128 at 3/3: 5.2 + 5.7 us with 12, 5.7 + 6.3 with 16, 7.0 + 7.8 with 8
// waves of 4 rows; 1090x436 at 2/2: 6.0 + 6.6 us with 16 against 7.1 + 7.7
// with 12, whose 370 tiles exceed the CUs).  Up to four per CU: 8 waves of 4
// rows, so that several workgroups share a CU and one loads while another
// computes (1280x720 at 3/3: 10.4 + 10.0 us against 11.3 + 11.4 us with 8
// waves of 6 rows and 11.1 + 9.7 us with 16 of 2).  Above: 8 waves of 6 rows,
// whose halo rows are a smaller share (4096x2048 at 2/2: 33.6 + 31.2 us
// against 38.5 + 35.5 us with 8 rows, whose fewer workgroups overlap less;
// 3072x1536 at 3/3: 29.2 + 27.0 us against 32.6 + 28.9 us with 4).
template <int NU> using RegTileTiny = RegTile<NU, 2, 12>;
template <int NU> using RegTileSmall = RegTile<NU, 2, 16>;
template <int NU> using RegTileMid = RegTile<NU, 4, 8>;
template <int NU> using RegTileBig = RegTile<NU, 6, 8>;
enum PassShape { PASS_TINY, PASS_SMALL, PASS_MID, PASS_BIG };
constexpr long kPassCUs = 256;
// tiny_tiles, small_tiles: tiles of the two small shapes (Mid has as many as Small)
inline PassShape pass_shape(long tiny_tiles, long small_tiles) {
  if (tiny_tiles <= kPassCUs) return PASS_TINY;
  if (small_tiles <= kPassCUs) return PASS_SMALL;
  return small_tiles <= 4 * kPassCUs ? PASS_MID : PASS_BIG;
}
// fn(shape's RegTile<NU>{})
template <int NU, class Fn> void with_pass_shape(PassShape shape, Fn fn) {
  if (shape == PASS_TINY) fn(RegTileTiny<NU>{});
  else if (shape == PASS_SMALL) fn(RegTileSmall<NU>{});
  else if (shape == PASS_MID) fn(RegTileMid<NU>{});
  else fn(RegTileBig<NU>{});
}
template <class Fn> void with_pass(PassShape shape, int nu, Fn fn) {
  switch (nu) {
  case 0: with_pass_shape<0>(shape, fn); break;
  case 1: with_pass_shape<1>(shape, fn); break;
  case 2: with_pass_shape<2>(shape, fn); break;
  default: with_pass_shape<3>(shape, fn); break;
  }
}
// the largest tile a shape's pass owns
inline void pass_tile(PassShape shape, bool pre, int nu, int *otx, int *oty) {
  with_pass(shape, nu, [&](auto t) {
    using T = decltype(t);
    *otx = pre ? T::OTXP : T::OTXQ;
    *oty = pre ? T::OTYP : T::OTYQ;
  });
}

// a tile's registers and its place in the level
template <class T> struct TileRegs {
  static constexpr int CPL = T::CPL, RPW = T::RPW, WAVES = T::WAVES;
  float P[RPW][CPL], F[RPW][CPL];
  unsigned M[RPW];                 // mask bytes of the lane's cells
  float below[CPL], above[CPL];    // the rows next to the wave's
  HeldRule rule[T::HOLD ? RPW : 1][CPL];
  const uint4 *tab;
  float *xb;                       // exchange buffers
  int w, h, lane, wave, x0, y0;    // x0: the lane's first column, y0: the wave's first row
  unsigned xs;                     // x0 clamped so that the lane's loads stay in the row
  unsigned ok, fast;               // rows in the interior / uniform (bit i: row i)
  bool edge, zgx, zgy;             // the region reaches outside the interior columns / a
                                   // side column / the wave holds or meets row 0 or h-1
  bool straight;                   // every row uniform and every column interior
  bool xin[CPL];                   // the cell's column is interior

  __device__ __forceinline__ void place(char *smem, int gx0, int gy0, int w_, int h_) {
    tab = (const uint4 *)smem;
    xb = (float *)(smem + T::TAB);
    w = w_;
    h = h_;
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    x0 = gx0 + CPL * lane;
    y0 = gy0 + RPW * wave;
    xs = (unsigned)min(max(x0, 0), w - CPL);
    edge = gx0 < 1 || gx0 + T::COLS > w - 1;
    zgx = gx0 < 1 || gx0 + T::COLS >= w;
    zgy = y0 <= 0 || y0 + RPW >= h - 1;
#pragma unroll
    for (int c = 0; c < CPL; c++) xin[c] = x0 + c >= 1 && x0 + c <= w - 2;
  }
  // one row of a field: a vector load at a column clamped into the row
  __device__ __forceinline__ void load_row(float (&v)[CPL], const float *base, int y) const {
    const float *row = base + (size_t)min(max(y, 0), h - 1) * w;
    const pair_u q = *(const pair_u *)((const char *)row + 4u * xs);
#pragma unroll
    for (int c = 0; c < CPL; c++) v[c] = q[c];
  }
  __device__ __forceinline__ unsigned load_mask_row(const uint8_t *base, int y) const {
    const uint8_t *row = base + (size_t)min(max(y, 0), h - 1) * w;
    return *(const mpair_u *)(row + xs);
  }
  // Where the clamp moved the last column's pair of an odd-width level, the
  // column goes to its place (cells outside the level hold values that no
  // interior cell uses).
  __device__ __forceinline__ bool shifted() const { return edge && w % 2 != 0; }
  __device__ __forceinline__ void shift(float (&v)[CPL]) const {
    v[0] = x0 - (int)xs == 1 ? v[1] : v[0];
  }
  __device__ __forceinline__ void shift_tile(bool p_too) {
#pragma unroll
    for (int i = 0; i < RPW; i++) {
      if (p_too) shift(P[i]);
      shift(F[i]);
      M[i] = x0 - (int)xs == 1 ? M[i] >> 8 : M[i];
    }
  }

  // the row bits, after the masks
  __device__ __forceinline__ void classify(float alpha) {
    constexpr unsigned full = 0x9f9fu; // both cells and their neighbours fluid
    unsigned keep = 0u; // mask bytes of interior columns
#pragma unroll
    for (int c = 0; c < CPL; c++) keep |= xin[c] ? 0xffu << (8 * c) : 0u;
    ok = fast = 0u;
#pragma unroll
    for (int i = 0; i < RPW; i++) {
      const bool in = y0 + i >= 1 && y0 + i <= h - 2;
      const bool uni = __ballot(((M[i] ^ full) & keep) != 0u) == 0ull;
      ok |= in ? 1u << i : 0u;
      fast |= in && uni && alpha == 1.0f ? 1u << i : 0u;
    }
    ok = __builtin_amdgcn_readfirstlane(ok);
    fast = __builtin_amdgcn_readfirstlane(fast);
    straight = !edge && fast == (1u << RPW) - 1u;
    if (T::HOLD && !straight) {
      stay_branch();
#pragma unroll
      for (int i = 0; i < (T::HOLD ? RPW : 0); i++)
#pragma unroll
        for (int c = 0; c < CPL; c++) rule[i][c] = held_rule(mask_of(i, c));
    }
  }

  __device__ __forceinline__ unsigned mask_of(int i, int c) const { return (M[i] >> (8 * c)) & 0xffu; }
  __device__ __forceinline__ float west(int i, int c) const {
    return c > 0 ? P[i][c > 0 ? c - 1 : 0] : lane_left(P[i][CPL - 1]);
  }
  __device__ __forceinline__ float east(int i, int c) const {
    return c < CPL - 1 ? P[i][c < CPL - 1 ? c + 1 : c] : lane_right(P[i][0]);
  }
  __device__ __forceinline__ float south(int i, int c) const {
    return i > 0 ? P[i > 0 ? i - 1 : 0][c] : below[c];
  }
  __device__ __forceinline__ float north(int i, int c) const {
    return i < RPW - 1 ? P[i < RPW - 1 ? i + 1 : i][c] : above[c];
  }

  __device__ __forceinline__ float relaxed(int i, int c, float hh) const { // uniform row
    float v = 0.0f;
    v += west(i, c);
    v += east(i, c);
    v += south(i, c);
    v += north(i, c);
    v += F[i][c] * hh * hh;
    v *= 0.25f;                                // = v / 4
    v = __builtin_fmaf(v, 0.0f, v);            // v, NaN for an infinite one
    return __builtin_fmaf(P[i][c], 0.0f, v);   // 1 v + 0 p
  }
  // colour phase: the cells with (c + i) & 1 == S
  template <int S> __device__ __forceinline__ void phase(float hh, float alpha) {
    if (straight) {
#pragma unroll
      for (int i = 0; i < RPW; i++)
#pragma unroll
        for (int c = (S + i) & 1; c < CPL; c += 2) P[i][c] = relaxed(i, c, hh);
      return;
    }
    if (T::HOLD) {
      stay_branch();
#pragma unroll
      for (int i = 0; i < RPW; i++)
#pragma unroll
        for (int c = (S + i) & 1; c < CPL; c += 2) {
          const float v = smooth_held(P[i][c], west(i, c), east(i, c), south(i, c), north(i, c),
                                      F[i][c] * hh * hh, rule[T::HOLD ? i : 0][c], alpha);
          P[i][c] = xin[c] && ((ok >> i) & 1u) ? v : P[i][c];
        }
      return;
    }
#pragma unroll
    for (int i = 0; i < RPW; i++) {
      if ((fast >> i) & 1u) {
#pragma unroll
        for (int c = (S + i) & 1; c < CPL; c += 2) {
          const float v = relaxed(i, c, hh);
          P[i][c] = xin[c] ? v : P[i][c];
        }
      } else if ((ok >> i) & 1u) {
        stay_branch();
#pragma unroll
        for (int c = (S + i) & 1; c < CPL; c += 2) {
          const float v = smooth_tab(P[i][c], west(i, c), east(i, c), south(i, c), north(i, c),
                                     F[i][c] * hh * hh, tab, mask_of(i, c), alpha);
          P[i][c] = xin[c] ? v : P[i][c];
        }
      }
    }
  }
  // publish / fetch the cells of colour S in the wave's first and last row;
  // a buffer is written again three exchanges later, when every wave has
  // passed the barriers after its reads
  __device__ __forceinline__ float *slot(int buf, int v, int last) const {
    return xb + buf * T::XBUF + (v * 2 + last) * T::XROW + lane;
  }
  template <int S> __device__ __forceinline__ void publish(int buf) {
    *slot(buf, wave, 0) = P[0][S];
    *slot(buf, wave, 1) = P[RPW - 1][1 - S];
  }
  template <int S> __device__ __forceinline__ void fetch(int buf) {
    if (wave > 0) below[1 - S] = *slot(buf, wave - 1, 1);
    if (wave < WAVES - 1) above[S] = *slot(buf, wave + 1, 0);
  }
  // setZeroGradientBC on the region: side columns of the interior rows, then
  // rows 0 and h-1 over the interior columns.  Rows 0 and 1 share a wave (its
  // first row is even); row h-1 may be a wave's first row, whose row below is
  // then `below`, and the wave of row h-2 sees the copy in `above`.
  __device__ __forceinline__ void zero_gradient() {
    if (zgx) {
      stay_branch();
#pragma unroll
      for (int i = 0; i < RPW; i++) {
        const float left = lane_left(P[i][CPL - 1]);
        const bool row = (ok >> i) & 1u;
#pragma unroll
        for (int c = 0; c < CPL; c++)
          P[i][c] = row && x0 + c == w - 1 ? (c > 0 ? P[i][c > 0 ? c - 1 : 0] : left) : P[i][c];
        P[i][0] = row && x0 == 0 ? P[i][1] : P[i][0];
      }
    }
    if (zgy) {
      stay_branch();
#pragma unroll
      for (int i = 0; i < RPW; i++)
#pragma unroll
        for (int c = 0; c < CPL; c++) {
          if (i % 2 == 0) P[i][c] = xin[c] && y0 + i == 0 ? P[i + 1 < RPW ? i + 1 : i][c] : P[i][c];
          P[i][c] = xin[c] && y0 + i == h - 1 ? south(i, c) : P[i][c];
        }
#pragma unroll
      for (int c = 0; c < CPL; c++)
        above[c] = xin[c] && y0 + RPW - 1 == h - 2 ? P[RPW - 1][c] : above[c];
    }
  }
  // NU sweeps; LAST: the rows next to the wave's are current at the end
  template <bool ZG, bool LAST>
  __device__ __forceinline__ void sweeps(float hh, float alpha, int &buf) {
#pragma unroll 1
    for (int s = 0; s < T::NU; s++) {
      phase<1>(hh, alpha);
      publish<1>(buf);
      __syncthreads();
      fetch<1>(buf);
      buf = buf == 2 ? 0 : buf + 1;
      phase<0>(hh, alpha);
      if (LAST || ZG || s + 1 < T::NU) {
        publish<0>(buf);
        __syncthreads();
        fetch<0>(buf);
        buf = buf == 2 ? 0 : buf + 1;
      }
      if (ZG) zero_gradient();
    }
  }
  // the owned cells
  __device__ __forceinline__ void store(float *out, int X0, int Y0, int otx, int oty) const {
    const int x1 = min(X0 + otx, w), y1 = min(Y0 + oty, h);
    const bool own = x0 >= X0 && x0 < x1, whole = x0 + CPL <= x1;
#pragma unroll
    for (int i = 0; i < RPW; i++) {
      const int y = y0 + i;
      if (y < Y0 || y >= y1) continue;
      float *row = out + (size_t)y * w;
      if (own && whole) {
        pair_u q;
#pragma unroll
        for (int c = 0; c < CPL; c++) q[c] = P[i][c];
        *(pair_u *)(row + (unsigned)x0) = q;
      } else if (own) {
#pragma unroll
        for (int c = 0; c < CPL; c++)
          if (x0 + c < x1) row[x0 + c] = P[i][c];
      }
    }
  }
};

// Pre-smoothing + calculateResidualField + restrict (pressure_solver.cpp:
// 213-227) of the tile at (X0, Y0): otx <= OTXP and oty <=
// OTYP, both even; X0 and Y0 are multiples of otx and oty.  Reads p (ZP: p is
// zero on entry and is not read), writes the smoothed level to p_out, the
// coarse rhs to fc and, unless ec is null, zero to the coarse solution's
// interior.
template <class T, bool ZP, bool ZG>
__device__ __forceinline__ void
regtile_pre(char *smem, int X0, int Y0, int otx, int oty, const float *__restrict__ p,
            float *__restrict__ p_out, const float *__restrict__ f,
            const uint8_t *__restrict__ m, int w, int h, float hh, float alpha, float ihsq,
            float *__restrict__ fc, float *__restrict__ ec, int wc, int hc) {
  constexpr int CPL = T::CPL, RPW = T::RPW;
  TileRegs<T> t;
  t.place(smem, X0 - T::HXP, Y0 - T::HYP, w, h);
#pragma unroll
  for (int i = 0; i < RPW; i++) {
    t.M[i] = t.load_mask_row(m, t.y0 + i);
    if (!ZP) t.load_row(t.P[i], p, t.y0 + i);
    t.load_row(t.F[i], f, t.y0 + i);
  }
  if (!ZP) {
    t.load_row(t.below, p, t.y0 - 1);
    t.load_row(t.above, p, t.y0 + RPW);
  } else {
#pragma unroll
    for (int c = 0; c < CPL; c++) {
      t.below[c] = t.above[c] = 0.0f;
#pragma unroll
      for (int i = 0; i < RPW; i++) t.P[i][c] = 0.0f;
    }
  }
  if (!T::HOLD) {
    fill_rule_table((uint4 *)smem);
    __syncthreads();
  }
  if (t.shifted()) {
    stay_branch();
    t.shift_tile(!ZP);
    if (!ZP) {
      t.shift(t.below);
      t.shift(t.above);
    }
  }
  t.classify(alpha);
  int buf = 0;
  t.template sweeps<ZG, true>(hh, alpha, buf);
  t.store(p_out, X0, Y0, otx, oty);
  // the residual in place of f
  auto uniform_residual = [&](int i, int c) {
    float v = 0.0f;
    v += t.west(i, c);
    v += t.east(i, c);
    v += t.south(i, c);
    v += t.north(i, c);
    v += -4.0f * t.P[i][c]; // the product apart: it may overflow where the sum would not
    v *= ihsq;
    return t.F[i][c] + v;
  };
  if (t.straight) {
#pragma unroll
    for (int i = 0; i < RPW; i++)
#pragma unroll
      for (int c = 0; c < CPL; c++) t.F[i][c] = uniform_residual(i, c);
  } else {
#pragma unroll
    for (int i = 0; i < RPW; i++) {
      if ((t.fast >> i) & 1u) {
#pragma unroll
        for (int c = 0; c < CPL; c++) t.F[i][c] = uniform_residual(i, c);
      } else if ((t.ok >> i) & 1u) {
        stay_branch();
#pragma unroll
        for (int c = 0; c < CPL; c++)
          t.F[i][c] = residual_of(t.P[i][c], t.west(i, c), t.east(i, c), t.south(i, c),
                                  t.north(i, c), t.F[i][c], t.mask_of(i, c), ihsq);
      }
    }
  }
  // the row below the wave's first one
  float rb[CPL];
  {
    float *mine = t.xb + buf * T::XBUF + t.wave * 2 * T::XROW + t.lane * CPL;
#pragma unroll
    for (int c = 0; c < CPL; c++) mine[c] = t.F[RPW - 1][c];
    __syncthreads();
    const float *from = t.wave > 0 ? mine - 2 * T::XROW : mine;
#pragma unroll
    for (int c = 0; c < CPL; c++) rb[c] = from[c];
  }
  // restrict (pressure_solver.cpp:118-132): coarse cells whose centre
  // (2X, 2Y) lies in the tile
  const int cx0 = max(X0 >> 1, 1), cx1 = min((X0 + otx) >> 1, wc - 1);
  const int cy0 = max(Y0 >> 1, 1), cy1 = min((Y0 + oty) >> 1, hc - 1);
#pragma unroll
  for (int i = 0; i < RPW; i += 2) {
    const int Y = (t.y0 + i) >> 1;
    if (Y < cy0 || Y >= cy1) continue;
    float lo[CPL], l0, l1, l2;
#pragma unroll
    for (int c = 0; c < CPL; c++) lo[c] = i > 0 ? t.F[i > 0 ? i - 1 : 0][c] : rb[c];
    l0 = lane_left(lo[CPL - 1]);
    l1 = lane_left(t.F[i][CPL - 1]);
    l2 = lane_left(t.F[i + 1][CPL - 1]);
#pragma unroll
    for (int c = 0; c < CPL; c += 2) {
      const float a0 = c > 0 ? lo[c > 0 ? c - 1 : 0] : l0;
      const float a1 = c > 0 ? t.F[i][c > 0 ? c - 1 : 0] : l1;
      const float a2 = c > 0 ? t.F[i + 1][c > 0 ? c - 1 : 0] : l2;
      float v = 0.0f;
      v = a0 * 1.0f + lo[c] * 2.0f + lo[c + 1] * 1.0f;
      v += a1 * 2.0f + t.F[i][c] * 4.0f + t.F[i][c + 1] * 2.0f;
      v += a2 * 1.0f + t.F[i + 1][c] * 2.0f + t.F[i + 1][c + 1] * 1.0f;
      const int X = (t.x0 + c) >> 1;
      if (X >= cx0 && X < cx1) {
        const size_t ci = (size_t)Y * wc + X;
        fc[ci] = v * (1.0f / 16.0f);
        if (ec) ec[ci] = 0.0f;
      }
    }
  }
}

// prolongate + correct (pressure_solver.cpp:134-181) + post-smoothing of the
// tile at (X0, Y0) (otx <= OTXQ, oty <= OTYQ): reads p and the coarse
// solution ec with its mask mc, writes p_out.
template <class T, bool ZG>
__device__ __forceinline__ void
regtile_post(char *smem, int X0, int Y0, int otx, int oty, const float *__restrict__ p,
             float *__restrict__ p_out, const float *__restrict__ f,
             const uint8_t *__restrict__ m, int w, int h, float hh, float alpha,
             const float *__restrict__ ec, const uint8_t *__restrict__ mc, int wc, int hc) {
  constexpr int CPL = T::CPL, RPW = T::RPW, CR = RPW / 2 + 1, CC = CPL / 2;
  TileRegs<T> t;
  // under ZG a tile that owns only the last column or row copies the one
  // before it, which has to be exact too
  t.place(smem, X0 - T::HXQ - (ZG && X0 == w - 1 ? CPL : 0),
          Y0 - T::HYQ - (ZG && Y0 == h - 1 ? 2 : 0), w, h);
  // coarse rows y0/2 .. y0/2 + RPW/2 under the wave's rows, coarse columns
  // x0/2 .. x0/2 + CPL/2 under the lane's (clamped: values outside the level
  // reach no corrected cell), the last from the lane to the right
  float E[CR][CC + 1];
  int G[CR][CC + 1];
  const int X = t.x0 >> 1, Yb = t.y0 >> 1;
#pragma unroll
  for (int i = 0; i < RPW; i++) {
    t.M[i] = t.load_mask_row(m, t.y0 + i);
    t.load_row(t.P[i], p, t.y0 + i);
  }
#pragma unroll
  for (int k = 0; k < CR; k++) {
    const size_t ro = (size_t)min(max(Yb + k, 0), hc - 1) * wc;
#pragma unroll
    for (int a = 0; a < CC; a++) {
      const unsigned xa = (unsigned)min(max(X + a, 0), wc - 1);
      E[k][a] = (ec + ro)[xa];
      G[k][a] = (mc + ro)[xa] & MK_SELF;
    }
  }
#pragma unroll
  for (int i = 0; i < RPW; i++) t.load_row(t.F[i], f, t.y0 + i);
  if (!T::HOLD) {
    fill_rule_table((uint4 *)smem);
    __syncthreads();
  }
  if (t.shifted()) {
    stay_branch();
    t.shift_tile(true);
  }
  t.classify(alpha);
  // coarse rows whose cells are all fluid (bit k)
  unsigned call = 0u;
#pragma unroll
  for (int k = 0; k < CR; k++) {
    bool all = true;
#pragma unroll
    for (int a = 0; a < CC; a++) all = all && G[k][a] != 0;
    call |= __ballot(!all) == 0ull ? 1u << k : 0u;
    E[k][CC] = lane_right(E[k][0]);
    G[k][CC] = __float_as_int(lane_right(__int_as_float(G[k][0])));
  }
  // fine and coarse flags 1: the divisors are constants
  auto uniform_e = [&](int i, int c) {
    const int k = i / 2, a = c / 2;
    if (i % 2 == 0 && c % 2 == 0) return E[k][a];
    if (i % 2 == 0) return (E[k][a] + E[k][a + 1]) / eps_count(2);
    const int k1 = k + 1 < CR ? k + 1 : k;
    if (c % 2 == 0) return (E[k][a] + E[k1][a]) / eps_count(2);
    return (E[k][a] + E[k1][a + 1] + E[k][a + 1] + E[k1][a]) / eps_count(4);
  };
  if (t.straight && t.y0 + RPW <= h - 2 && call == (1u << CR) - 1u) {
#pragma unroll
    for (int i = 0; i < RPW; i++)
#pragma unroll
      for (int c = 0; c < CPL; c++) t.P[i][c] += uniform_e(i, c);
  } else {
#pragma unroll
    for (int i = 0; i < RPW; i++) {
      const int k = i / 2, k1 = k + 1 < CR ? k + 1 : k;
      // an odd row needs the coarse row above
      if (!((t.ok >> i) & 1u) || (i % 2 == 1 && t.y0 + i > h - 3)) continue;
      stay_branch();
      if (((t.fast >> i) & 1u) && ((call >> k) & 1u) && (i % 2 == 0 || ((call >> k1) & 1u))) {
#pragma unroll
        for (int c = 0; c < CPL; c++) {
          const float v = t.P[i][c] + uniform_e(i, c);
          t.P[i][c] = t.xin[c] && (c % 2 == 0 || t.x0 + c <= w - 3) ? v : t.P[i][c];
        }
      } else {
        stay_branch();
#pragma unroll
        for (int c = 0; c < CPL; c++) {
          const int a = c / 2;
          const float Fs = (t.mask_of(i, c) & MK_SELF) ? 1.0f : 0.0f;
          float e;
          if (i % 2 == 0 && c % 2 == 0) e = E[k][a] * Fs;
          else if (i % 2 == 0) e = Fs * (E[k][a] + E[k][a + 1]) / eps_count(G[k][a] + G[k][a + 1]);
          else if (c % 2 == 0) e = Fs * (E[k][a] + E[k1][a]) / eps_count(G[k][a] + G[k1][a]);
          else
            e = Fs * (E[k][a] + E[k1][a + 1] + E[k][a + 1] + E[k1][a]) /
                eps_count(G[k][a] + G[k1][a + 1] + G[k][a + 1] + G[k1][a]);
          t.P[i][c] = t.xin[c] && (c % 2 == 0 || t.x0 + c <= w - 3) ? t.P[i][c] + e : t.P[i][c];
        }
      }
    }
  }
  int buf = 0;
  if (T::NU > 0 || ZG) {
    // both colours of the wave's first and last row
#pragma unroll
    for (int c = 0; c < CPL; c++) t.below[c] = t.above[c] = 0.0f;
    t.template publish<1>(0);
    t.template publish<0>(1);
    __syncthreads();
    t.template fetch<1>(0);
    t.template fetch<0>(1);
    buf = 2;
    if (ZG) t.zero_gradient();
    t.template sweeps<ZG, false>(hh, alpha, buf);
  }
  t.store(p_out, X0, Y0, otx, oty);
}

} // namespace ubg
