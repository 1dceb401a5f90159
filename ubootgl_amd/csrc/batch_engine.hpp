// batch_engine.hpp -- internal to libubg.so: the engine that advances many
// independent refinement solves together (batched and served solves).
//
// Layout: every domain owns, from a device arena, the float64 solution x
// (two buffers), its float32 rhs, the FP32 V-cycle buffers of the levels down
// to the first one solved in LDS (p twice, f) and its solve state; the flag
// and mask pyramid (a "geometry") can be shared by domains of the same shape.
// The engine keeps device tables of the current member domains and, per
// step, a row of per-domain buffer indices for every stage, so that one
// launch of a stage serves every domain whatever its level count.
#pragma once

#include "capi_common.hpp"
#include "coarse_device.hpp"
#include "regtile_device.hpp"

#include <map>
#include <memory>

namespace ubg {

constexpr int BMAXL = 16;        // levels per domain at most
constexpr int B_UPD_W = 256;     // update tile: 256 x 8 cells, as the
constexpr int B_UPD_H = 8;       //   single-domain refinement's blocks
constexpr int B_MIN_SIZE = 16;

// solve state of one domain (device; written by the norm kernel)
struct DState {
  double r0, rel, best, tol;
  double ref; // > 0: residuals are relative to ref, not to the first one
  int active, converged, iters, vcycles, stall, max_iter, xcur, k;
  int nonfinite, pad;
  double hist[UBG_IR_HISTORY];
};

// device table rows
struct BLev {
  float *p[2];
  float *f;
  const uint8_t *mask;
  int w, h;
  float hh, ihsq;
};
struct BDom {
  DState *st;
  double *x[2];
  const float *rhs;
  double *partial;
  int w, h, gx, gy, nlev, cfirst;
};
struct Tile {
  int d, x0, y0, i;
};

// first-fit device sub-allocator over one hipMalloc (256-byte granules)
class Arena {
public:
  int init(size_t bytes);
  void release();
  char *alloc(size_t bytes); // nullptr if it does not fit
  void free(char *p);
  size_t capacity() const { return cap_; }
  size_t used() const { return used_; }
  char *base() const { return base_; }

private:
  char *base_ = nullptr;
  size_t cap_ = 0, used_ = 0;
  std::map<size_t, size_t> free_; // offset -> size
  std::map<size_t, size_t> live_; // offset -> size
};

// flag/mask pyramid of one domain shape (device, read-only once built)
struct BGeom {
  int W = 0, H = 0, nlev = 0, cfirst = 0;
  int w[BMAXL] = {}, h[BMAXL] = {};
  uint8_t *flag[BMAXL] = {}, *mask[BMAXL] = {};
  char *mem = nullptr;
  size_t bytes = 0;
  size_t lds_bytes = 0;
  int refs = 0;
  bool ring_fluid = false; // every outer-ring cell is fluid
};

struct BDomain {
  uint64_t id = 0; // no two domains of an engine have the same
  BGeom *g = nullptr;
  float h = 0.0f;
  float hh[BMAXL] = {};
  float *p[BMAXL][2] = {};
  float *f[BMAXL] = {};
  double *x[2] = {};
  float *rhs = nullptr;
  double *partial = nullptr;
  DState *st = nullptr;
  int gx = 0, gy = 0;
  char *mem = nullptr;
  size_t bytes = 0;
  // host copy of the buffer indices (which p of each level, which x is current)
  int cur[BMAXL] = {};
  int xcur = 0;
};

struct Tuning {
  int tx = 64, ty = 8, blocks = 0; // smoother tile (sweep stages), workgroups per launch
  int prow = 0;                    // tile shape of the level passes (0: chosen per level)
};

// Level sizes, first LDS level and byte counts of a W x H domain.
struct BShape {
  int nlev = 0, cfirst = 0;
  int w[BMAXL] = {}, h[BMAXL] = {};
  size_t lds_bytes = 0, geom_bytes = 0, dom_bytes = 0;
};
int batch_shape(int W, int H, BShape *s);

// An engine's small memory: pinned host blocks with device blocks of the same
// sizes, carved in pairs and kept until the engine ends.  One block made with
// the engine holds what its members need; where they outgrow it, another at
// least as large as those before it is added.  (A pair of allocations costs 175
// us and its release as much, so sixteen of them, made by the first solves,
// took a new server's first burst of four 32x32 requests from 1.7 to 2.4 ms and
// the destruction of a batch of eight from 0.1 to 1.2 ms.)
class Staging {
public:
  ~Staging();
  int reserve(size_t bytes); // the next `bytes` come from one block
  int carve(size_t bytes, char **host, char **dev);

private:
  struct Block {
    char *host = nullptr, *dev = nullptr;
    size_t cap = 0, used = 0;
  };
  std::vector<Block> blocks_;
};

// Host tables on their way to the device: two slots, used in turn, so that a
// table is prepared while the work that reads the one before it runs.  A
// slot's device copy belongs to the work queued between its put and the next;
// it is written again once that work has passed.  (Solves and server turns end
// with a synchronisation, so the slots' events have passed when they are waited
// for.)
class UploadRing {
public:
  static constexpr int SLOTS = 2;
  ~UploadRing();
  int reserve(Staging &st, size_t bytes);
  int put(Staging &st, const void *data, size_t bytes, hipStream_t s, char **dev);

private:
  struct Slot {
    char *host = nullptr, *dev = nullptr;
    size_t cap = 0;
    hipEvent_t used = nullptr; // recorded behind the slot's users
  } slot_[SLOTS];
  int cur_ = -1;
};

class BatchEngine {
public:
  ~BatchEngine();
  // members: how many domains to have tables for at once (more are allocated
  // when they come)
  int init(hipStream_t s, const ubg_params &prm, int vcycles_per_step, int members);
  hipStream_t stream() const { return stream_; }
  const ubg_params &params() const { return prm_; }
  int vcycles() const { return k_; }
  // levels run as the pre / post passes (smoothing counts that they take)
  bool tiled() const { return prm_.nu_pre <= kNuPass && prm_.nu_post <= kNuPass; }
  void set_vcycles(int k) {
    if (k != k_) drop_graphs();
    k_ = k;
  }

  // geometry / domain lifetime (memory from `arena`)
  // need_ring: the outer ring must be fluid (refinement solves hold it as
  // Dirichlet data); projection domains take any flag
  int geom_create(Arena &arena, int W, int H, const float *flag_host, BGeom **out,
                  bool need_ring = true);
  void geom_release(Arena &arena, BGeom *g);
  // The domain calls take an optional stream (default: the engine's own).
  // A caller that keeps a step in flight on the engine's stream may use
  // another stream for domains that are not members of that step.
  int domain_create(Arena &arena, BGeom *g, float h, BDomain **out, hipStream_t s = nullptr);
  void domain_release(Arena &arena, BDomain *d);
  int domain_set_rhs(BDomain *d, const float *rhs_host);
  int domain_set_guess(BDomain *d, const double *x_host);
  // reset a domain's solve state: active, tol/max_iter, fresh (next update
  // computes r0 and does not add e)
  int domain_start(BDomain *d, double tol, int max_iter, double ref = 0.0,
                   hipStream_t s = nullptr);
  int domain_read_state(BDomain *d, DState *out, hipStream_t s = nullptr);
  // the same for several domains at once, on the engine's stream
  int start_all(const std::vector<BDomain *> &doms, double tol, int max_iter);
  int read_states(const std::vector<BDomain *> &doms, std::vector<DState> &out);
  int domain_get_solution(BDomain *d, double *x_host, hipStream_t s = nullptr);
  // level-0 pressure and rhs of the plain V-cycles (projection solves); kind
  // is a hipMemcpyKind (host or device arrays); p == nullptr clears p
  int domain_set_level0(BDomain *d, const float *p, const float *f, hipMemcpyKind kind,
                        hipStream_t s = nullptr);
  int domain_get_pressure(BDomain *d, float *p, hipMemcpyKind kind, hipStream_t s = nullptr);

  // the member set of the following steps: `running` domains take V-cycles
  // and an accumulating update; `fresh` ones only their first update
  int set_members(const std::vector<BDomain *> &running, const std::vector<BDomain *> &fresh);
  // forget the member set (a member domain is about to be released, or the
  // tables could not be built), so the next set_members rebuilds the tables
  void invalidate_members() {
    run_.clear();
    fresh_.clear();
    all_.clear();
    ids_.clear();
    d_lev_ = nullptr;
    drop_graphs();
  }
  // enqueue `nsteps` refinement steps of the members; the active-domain
  // count lands in *count_host (pinned) when the stream reaches it
  int enqueue_steps(int nsteps);
  // the same from a captured graph (no fresh members)
  int replay_steps(int nsteps);
  // the first update (r0, no V-cycles) of every member, as if all were fresh
  int enqueue_first_update();
  // ncycles plain FP32 V-cycles (MG::solve, pressure_solver.cpp:250-257) of
  // every running member on its level-0 pressure and rhs; zg: level 0 takes
  // setZeroGradientBC after every sweep and after the correction (the
  // simulation's projection); needs 1 <= nu_pre, nu_post <= kNuPass.
  int enqueue_vcycles(int ncycles, bool zg);
  int active_count() const { return *count_host_; }
  // members whose solve was still active at the last completed step
  std::vector<BDomain *> active_members() const;
  size_t members() const { return all_.size(); }
  int sync();

  int set_tuning(const Tuning &t);
  const Tuning &tuning() const { return tune_; }
  // time each compiled smoother tile shape and block count over the member
  // levels; keeps the fastest
  int autotune(double *best_ms);

private:
  struct StageRec {
    int kind, level;
    size_t off;
  };
  int build_tables();
  int reserve_active(size_t n);
  int build_tiles();
  void gen_steps(int nsteps, std::vector<StageRec> &st, std::vector<uint8_t> &idx,
                 bool all_fresh = false);
  void gen_vcycle_tiled(std::vector<StageRec> &st, std::vector<uint8_t> &idx);
  int launch_stages(const std::vector<StageRec> &st, const uint8_t *d_idx);
  int upload_idx(const std::vector<uint8_t> &idx, uint8_t **d_idx);
  int launch_sweeps_only(int reps);
  std::string state_key() const;

  hipStream_t stream_ = nullptr;
  ubg_params prm_{};
  int k_ = 4;
  Tuning tune_{};
  std::vector<BDomain *> run_, fresh_, all_;
  std::vector<uint64_t> ids_; // of all_, when the tables were built
  uint64_t next_id_ = 1;
  int lmax_ = 0;
  // device tables
  Staging staging_;
  UploadRing tab_ring_, off_ring_, idx_ring_, st_ring_;
  BLev *d_lev_ = nullptr; // in tab_ring_, as are d_dom_ and d_cargs_
  BDom *d_dom_ = nullptr;
  CoarseArgs *d_cargs_ = nullptr;
  size_t act_cap_ = 0;
  size_t coarse_lds_ = 0;
  bool coarse_big_ = false; // a member's first LDS level needs the larger variant
  // tile maps: per level sweep / rr / pc (running members), update (all):
  // prefix of tile counts over slots and tiles per row, in one int array
  std::vector<int> h_off_;
  int *d_off_ = nullptr; // in off_ring_
  struct Span {
    size_t off = 0; // into the int array
    int n = 0;      // tiles
    int nd = 0;     // domain slots covered
    int oty = 0;    // level passes: tile rows
    PassShape shape = PASS_SMALL; //   and shape
  };
  Span sw_[BMAXL], rr_[BMAXL], pc_[BMAXL], upd_;
  Span tp_[BMAXL], tq_[BMAXL]; // level passes (pre, post)
  bool zg0_ = false;            // the stages being launched apply ZG at level 0
  int launch_passes_only(int reps);
  int *d_count_ = nullptr;
  int *count_host_ = nullptr;
  uint8_t *d_active_ = nullptr; // per slot, written with the count
  uint8_t *h_active_ = nullptr; // pinned copy
  // graphs by index state (member sets that stay: projection batches, lone domains)
  struct Graph {
    hipGraphExec_t exec = nullptr;
    uint8_t *d_idx = nullptr;
  };
  std::map<std::string, Graph> graphs_;
  template <class Gen> int replay(const std::string &what, Gen gen);
  int capture(const std::vector<StageRec> &st, const std::vector<uint8_t> &idx, Graph *g);
  void drop_graphs();
};

} // namespace ubg
