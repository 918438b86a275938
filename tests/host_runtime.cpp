// A stand-in for the HIP runtime that runs no kernel, for CPU tests of what
// the library's host code asks of the runtime. Device memory is zeroed host
// memory (with a limit that a test can set), copies are copies, and every
// launch and stream wait is logged with its thread. Loaded with RTLD_GLOBAL
// before the library, so that its symbols are the ones the library binds to.
#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

namespace {
enum { OK = 0, NO_MEMORY = 2, UNKNOWN = 999 };
struct Dim3 {
  uint32_t x, y, z;
};
std::mutex mu;
std::map<const void *, std::string> kernels; // host stub -> device name
std::map<const void *, void *> symbols;      // host shadow of a device variable -> its memory
std::map<void *, size_t> blocks;             // device memory
size_t in_use = 0, limit = SIZE_MAX;
int launch_us = 0, fail_last_error = 0, last_error = OK, fill_copies = 0;
std::map<std::thread::id, int> threads;
std::string events;
void note(const char *what) { // (mu held)
  const int t = threads.emplace(std::this_thread::get_id(), (int)threads.size()).first->second;
  events += std::to_string(t) + " " + what + "\n";
}
} // namespace

extern "C" {
// ---- controls of the tests
void rt_memory_limit(size_t bytes) {
  std::lock_guard<std::mutex> l(mu);
  limit = bytes == SIZE_MAX ? SIZE_MAX : in_use + bytes;
}
size_t rt_in_use() { return in_use; }
void rt_launch_time(int us) { launch_us = us; }
void rt_fail_last_error(int n) { fail_last_error = n; }
void rt_fill_copies(int on) { fill_copies = on; }
size_t rt_events(char *buf, size_t len) {
  std::lock_guard<std::mutex> l(mu);
  const size_t n = events.size();
  if (buf && len > n) {
    std::memcpy(buf, events.c_str(), n + 1);
    events.clear();
  }
  return n;
}

// ---- the runtime
void **__hipRegisterFatBinary(const void *) {
  static void *module;
  return &module;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *stub, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
  kernels[stub] = name;
}
void __hipRegisterVar(void **, void *shadow, char *, const char *, int, size_t size, int, int) {
  symbols[shadow] = std::calloc(1, size);
}
int __hipPushCallConfiguration(Dim3, Dim3, size_t, void *) { return OK; }
int __hipPopCallConfiguration(Dim3 *g, Dim3 *b, size_t *shared, void **stream) {
  *g = *b = Dim3{1, 1, 1};
  *shared = 0;
  *stream = nullptr;
  return OK;
}
int hipLaunchKernel(const void *stub, Dim3, Dim3, void **, size_t, void *) {
  {
    std::lock_guard<std::mutex> l(mu);
    note(kernels.count(stub) ? kernels[stub].c_str() : "?");
  }
  if (launch_us) std::this_thread::sleep_for(std::chrono::microseconds(launch_us));
  return OK;
}
int hipMalloc(void **p, size_t n) {
  std::lock_guard<std::mutex> l(mu);
  if (in_use + n > limit) {
    *p = nullptr;
    return last_error = NO_MEMORY;
  }
  *p = std::calloc(1, n);
  blocks[*p] = n;
  in_use += n;
  return OK;
}
int hipFree(void *p) {
  std::lock_guard<std::mutex> l(mu);
  if (blocks.count(p)) in_use -= blocks[p];
  blocks.erase(p);
  std::free(p);
  return OK;
}
int hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::calloc(1, n);
  return OK;
}
int hipHostFree(void *p) {
  std::free(p);
  return OK;
}
int hipHostGetDevicePointer(void **d, void *h, unsigned) {
  *d = h;
  return OK;
}
int hipMemcpy(void *d, const void *s, size_t n, int) {
  std::memcpy(d, s, n);
  return OK;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int kind, void *) {
  std::memcpy(d, s, n);
  if (fill_copies && kind == 2) std::memset(d, 0xff, n); // what kernels would have left, device to host
  return OK;
}
int hipMemset(void *d, int v, size_t n) {
  std::memset(d, v, n);
  return OK;
}
int hipMemsetAsync(void *d, int v, size_t n, void *) {
  std::memset(d, v, n);
  return OK;
}
int hipGetDevice(int *d) {
  *d = 0;
  return OK;
}
int hipSetDevice(int) { return OK; }
int hipGetSymbolAddress(void **p, const void *shadow) {
  *p = symbols[shadow];
  return *p ? OK : UNKNOWN;
}
int hipGetLastError() {
  std::lock_guard<std::mutex> l(mu);
  if (fail_last_error > 0 && fail_last_error-- == 1) return UNKNOWN;
  const int e = last_error;
  last_error = OK;
  return e;
}
const char *hipGetErrorString(int e) { return e == NO_MEMORY ? "out of memory" : "unknown error"; }
int hipStreamCreateWithFlags(void **s, unsigned) {
  *s = std::malloc(1);
  return OK;
}
int hipStreamDestroy(void *s) {
  std::free(s);
  return OK;
}
int hipStreamQuery(void *) { return OK; }
int hipStreamSynchronize(void *) {
  std::lock_guard<std::mutex> l(mu);
  note("wait");
  return OK;
}
int hipStreamBeginCapture(void *, int) { return OK; }
int hipStreamEndCapture(void *, void **g) {
  *g = std::malloc(1);
  return OK;
}
int hipGraphInstantiate(void **e, void *, void **, char *, size_t) {
  *e = std::malloc(1);
  return OK;
}
int hipGraphUpload(void *, void *) { return OK; }
int hipGraphLaunch(void *, void *) { return OK; }
int hipGraphDestroy(void *g) {
  std::free(g);
  return OK;
}
int hipGraphExecDestroy(void *e) {
  std::free(e);
  return OK;
}
int hipEventCreate(void **e) {
  *e = std::malloc(1);
  return OK;
}
int hipEventDestroy(void *e) {
  std::free(e);
  return OK;
}
int hipEventRecord(void *, void *) { return OK; }
int hipEventSynchronize(void *) { return OK; }
int hipEventElapsedTime(float *ms, void *, void *) {
  *ms = 0.0f;
  return OK;
}
}
