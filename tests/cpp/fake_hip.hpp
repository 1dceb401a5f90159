// fake_hip.hpp -- stands in for the HIP runtime's memory, stream, event and
// launch calls of libubg.so in a program linked with -rdynamic: device memory is
// host memory and no kernel runs.  Allocations are counted and one of them can
// be made to fail; the sizes of the copies to the device are recorded.
#pragma once

#include <atomic>
#include <cstdlib>
#include <cstring>
#include <vector>

namespace {
constexpr int kOk = 0, kOutOfMemory = 2;
// the allocation to fail (0: none), allocations and releases so far
std::atomic<int> g_fail_at{0}, g_allocs{0}, g_frees{0};
std::vector<size_t> g_uploads; // sizes of the copies to the device
struct Dim {
  unsigned x, y, z;
};
Dim g_grid, g_block;
size_t g_shared;
void *g_stream;
int take(void **p, size_t n) {
  if (++g_allocs == g_fail_at) {
    *p = nullptr;
    return kOutOfMemory;
  }
  *p = std::calloc(1, n ? n : 1);
  return kOk;
}
} // namespace

extern "C" {
int hipGetDeviceCount(int *n) { return *n = 1, kOk; }
int hipGetDevice(int *d) { return *d = 0, kOk; }
int hipGetLastError() { return kOk; }
const char *hipGetErrorString(int e) { return e ? "out of memory" : "no error"; }
int hipMalloc(void **p, size_t n) { return take(p, n); }
int hipHostMalloc(void **p, size_t n, unsigned) { return take(p, n); }
int hipFree(void *p) { return g_frees++, std::free(p), kOk; }
int hipHostFree(void *p) { return g_frees++, std::free(p), kOk; }
int hipMemcpy(void *d, const void *s, size_t n, int) { return std::memcpy(d, s, n), kOk; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *) {
  if (kind == 1) g_uploads.push_back(n);
  return std::memcpy(d, s, n), kOk;
}
int hipMemset(void *d, int v, size_t n) { return std::memset(d, v, n), kOk; }
int hipMemsetAsync(void *d, int v, size_t n, void *) { return std::memset(d, v, n), kOk; }
int hipStreamCreateWithFlags(void **s, unsigned) { return *s = std::malloc(1), kOk; }
int hipStreamSynchronize(void *) { return kOk; }
int hipStreamDestroy(void *s) { return std::free(s), kOk; }
int hipEventCreate(void **e) { return *e = std::malloc(1), kOk; }
int hipEventCreateWithFlags(void **e, unsigned) { return *e = std::malloc(1), kOk; }
int hipEventRecord(void *, void *) { return kOk; }
int hipEventSynchronize(void *) { return kOk; }
int hipEventElapsedTime(float *ms, void *, void *) { return *ms = 1.0f, kOk; }
int hipEventDestroy(void *e) { return std::free(e), kOk; }
int hipFuncSetAttribute(const void *, int, int) { return kOk; }
int hipLaunchKernel(const void *, Dim, Dim, void **, size_t, void *) { return kOk; }
int __hipPushCallConfiguration(Dim g, Dim b, size_t n, void *s) {
  g_grid = g, g_block = b, g_shared = n, g_stream = s;
  return kOk;
}
int __hipPopCallConfiguration(Dim *g, Dim *b, size_t *n, void **s) {
  *g = g_grid, *b = g_block, *n = g_shared, *s = g_stream;
  return kOk;
}
}
