// A batched solve whose allocations fail: the program, with fake_hip.hpp in
// the HIP runtime's place, lets the k-th allocation of a call fail for every k,
// and checks that the call says so and that the next call uploads what a call
// after no failure uploads -- no table of an earlier member set or tuning is
// taken for the present one.  A handle allocates what it needs when it is
// made: solves, tunings and a server's ordinary bursts allocate and free
// nothing.  Runs without a GPU.
#include "fake_hip.hpp"

#include <ubg_c.h>

#include <cstdio>

namespace {
int g_bad = 0;
void expect(bool ok, const char *what, int k) {
  if (ok) return;
  std::printf("FAILED: %s (allocation %d fails; last error: %s)\n", what, k, ubg_last_error());
  g_bad++;
}

ubg_batch *make(int n, int side) {
  std::vector<int> w(n), h(n);
  for (int d = 0; d < n; d++) {
    w[d] = side + d;
    h[d] = side;
  }
  ubg_batch *b = nullptr;
  if (ubg_batch_create(n, w.data(), h.data(), nullptr, &b) != UBG_OK) std::exit(2);
  for (int d = 0; d < n; d++) {
    std::vector<float> one((size_t)w[d] * h[d], 1.0f);
    if (ubg_batch_set_domain(b, d, one.data(), one.data(), 0.1f) != UBG_OK) std::exit(2);
  }
  return b;
}

// no kernel runs, so a call that reaches its end finds no converged domain
bool reached_end(int rc) { return rc == UBG_E_NOT_CONVERGED; }

// `call` on a batch that `before` has been applied to, its k-th allocation
// failing for every k there is: the next solve's uploads are `want`, without
// the tables and tile maps only where the failed call uploaded both (after the
// states)
template <class Before, class Call>
void failing(const char *what, const std::vector<size_t> &want, Before before, Call call) {
  for (int k = 1;; k++) {
    ubg_batch *b = make(20, 40);
    before(b);
    g_allocs = 0;
    g_fail_at = k;
    g_uploads.clear();
    const int rc = call(b);
    const bool failed = g_allocs >= k, built = g_uploads.size() >= 3;
    g_fail_at = 0;
    if (failed) {
      expect(rc == UBG_E_OOM, what, k);
      g_uploads.clear();
      expect(reached_end(ubg_batch_solve(b, nullptr, nullptr)), what, k);
      const std::vector<size_t> rest = {want[0], want[3], want[4]};
      expect(g_uploads == want || (built && g_uploads == rest), "uploads after a failure", k);
    } else {
      std::printf("%s: %d allocations\n", what, k - 1);
    }
    ubg_batch_destroy(b);
    if (!failed) return;
  }
}
} // namespace

int main() {
  // uploads of a solve that builds its tables: states, tables, tile maps,
  // stage indices, states
  ubg_batch *b = make(20, 40);
  g_uploads.clear();
  expect(reached_end(ubg_batch_solve(b, nullptr, nullptr)), "solve", 0);
  const std::vector<size_t> want = g_uploads;
  expect(want.size() == 5, "uploads of a first solve", 0);
  ubg_batch_destroy(b);

  auto nothing = [](ubg_batch *) {};
  auto solve = [](ubg_batch *q) { return ubg_batch_solve(q, nullptr, nullptr); };
  // one of the domains replaced, so that the tables of the former solve are
  // another member set's
  auto replaced = [&](ubg_batch *q) {
    solve(q);
    std::vector<float> one((size_t)40 * 40, 1.0f);
    ubg_batch_set_domain(q, 0, one.data(), one.data(), 0.1f);
  };
  auto tune = [](ubg_batch *q) {
    ubg_batch_tuning t{};
    ubg_batch_get_tuning(q, &t);
    t.pass_rows = 8;
    return ubg_batch_set_tuning(q, &t);
  };
  failing("first solve", want, nothing, solve);
  failing("solve after a domain was replaced", want, replaced, solve);
  failing("a tuning after a solve", want, solve, tune);

  // 60 domains, two solves and a tuning
  b = make(60, 20);
  g_allocs = g_frees = 0;
  solve(b);
  tune(b);
  solve(b);
  expect(g_allocs == 0 && g_frees == 0, "allocations of solves", 0);
  ubg_batch_destroy(b);
  expect(g_frees <= 3, "releases of a batch", 0);

  // bursts of requests: two that a new server has tables for, larger ones, one
  // of them with an allocation that fails (its requests may fail, the next
  // ones do not)
  ubg_server_params sp;
  ubg_server_params_default(&sp);
  sp.hbm_budget = (size_t)64 << 20;
  ubg_server *srv = nullptr;
  if (ubg_server_create(&sp, nullptr, &srv) != UBG_OK) return 2;
  std::vector<float> one(24 * 20, 1.0f);
  int geom = 0;
  if (ubg_server_add_geometry(srv, 24, 20, one.data(), 0.1f, &geom) != UBG_OK) return 2;
  g_frees = 0;
  for (int n : {4, 60, 200, 500, 501}) {
    const float *rhs[2] = {one.data(), one.data()};
    const double fnorm[2] = {1.0, 1.0};
    std::vector<uint64_t> id(n);
    g_allocs = 0;
    g_fail_at = n == 500 ? 1 : 0;
    for (auto &i : id)
      if (ubg_server_submit(srv, geom, 2, rhs, fnorm, nullptr, &i) != UBG_OK) return 2;
    for (auto &i : id)
      expect(ubg_server_wait(srv, i, -1.0, nullptr) == UBG_OK || n == 500, "request", n);
    if (n <= 60) expect(g_allocs == 0, "allocations of a burst", n);
    expect(g_frees == 0, "releases in a burst", n);
    std::printf("burst of %d: %d allocations\n", n, (int)g_allocs);
  }
  ubg_server_destroy(srv);
  if (g_bad) return 1;
  std::printf("ALL OK\n");
  return 0;
}
