// A server's step takes the tables of its own members: a request that ends with
// its first update, then one on another geometry, whose domain may come to sit
// at the first one's address.  With fake_hip.hpp in the HIP runtime's place no
// kernel runs, so that every request ends with its first update.
#include "fake_hip.hpp"

#include <ubg_c.h>

#include <cstdio>

int main() {
  ubg_server_params sp;
  ubg_server_params_default(&sp);
  sp.hbm_budget = (size_t)64 << 20;
  ubg_server *s = nullptr;
  if (ubg_server_create(&sp, nullptr, &s) != UBG_OK) return 2;
  const int W[2] = {24, 40}, H[2] = {20, 33};
  std::vector<float> one[2];
  int geom[2];
  for (int g = 0; g < 2; g++) {
    one[g].assign((size_t)W[g] * H[g], 1.0f);
    if (ubg_server_add_geometry(s, W[g], H[g], one[g].data(), 0.1f, &geom[g]) != UBG_OK) return 2;
  }
  int bad = 0;
  for (int k = 0; k < 40; k++) {
    const int g = k % 2;
    const float *rhs = one[g].data();
    const double fnorm = 1.0;
    uint64_t id;
    g_uploads.clear();
    if (ubg_server_submit(s, geom[g], 1, &rhs, &fnorm, nullptr, &id) != UBG_OK) return 2;
    if (ubg_server_wait(s, id, -1.0, nullptr) != UBG_OK) return 2;
    // right-hand side, state, tables, tile maps, stage indices
    if (g_uploads.size() != 5) {
      std::printf("request %d: %zu uploads\n", k, g_uploads.size());
      bad++;
    }
  }
  ubg_server_destroy(s);
  if (bad) return 1;
  std::printf("ALL OK\n");
  return 0;
}
