// A stand-in for the HIP runtime, loaded ahead of it, so that the library's host
// code runs without a GPU: device memory is host memory, copies are made at
// once, launches are only written down, allocations fail on demand.
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <string>

namespace {
constexpr int OOM = 2, INVALID = 1;
size_t g_deny = SIZE_MAX;  // allocations of this many bytes or more fail
size_t g_deny_new = SIZE_MAX;  // those of the C++ code itself
int g_last = 0;
std::string g_log;
std::map<const void *, std::string> g_names;
std::map<char *, size_t> g_host;
struct Dim3 {
  uint32_t x, y, z;
};
struct Config {
  Dim3 grid, block;
  size_t shared;
  void *stream;
} g_config;
int g_token;
// what launches leave in memory, where a test needs it
double g_spacing = 0.0;
void (*g_hook)(const char *, void **) = nullptr;

int fail(int e) {
  g_last = e;
  return e;
}
int alloc(void **p, size_t n) {
  *p = nullptr;
  if (n >= g_deny) return fail(OOM);
  return n == 0 || (*p = calloc(1, n)) ? 0 : fail(OOM);
}
}  // namespace

void *operator new(size_t n) {
  void *p = n >= g_deny_new ? nullptr : malloc(n);
  if (!p) throw std::bad_alloc();
  return p;
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

extern "C" {

void fake_deny(size_t bytes) { g_deny = bytes; }
void fake_deny_new(size_t bytes) { g_deny_new = bytes; }
// the kernels launched so far, one a line
const char *fake_log() { return g_log.c_str(); }
void fake_clear() { g_log.clear(); }
// sheets this far apart, as the kernels that measure densities report them
void fake_spacing(double d) { g_spacing = d; }
// called with the name and the arguments of every launch
void fake_hook(void (*f)(const char *, void **)) { g_hook = f; }

void **__hipRegisterFatBinary(const void *) {
  static void *module;
  return &module;
}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, uint32_t,
                           void *, void *, void *, void *, int *) {
  g_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
int __hipPushCallConfiguration(Dim3 grid, Dim3 block, size_t shared, void *stream) {
  g_config = {grid, block, shared, stream};
  return 0;
}
int __hipPopCallConfiguration(Dim3 *grid, Dim3 *block, size_t *shared, void **stream) {
  *grid = g_config.grid;
  *block = g_config.block;
  *shared = g_config.shared;
  *stream = g_config.stream;
  return 0;
}
int hipLaunchKernel(const void *f, Dim3 grid, Dim3 block, void **args, size_t, void *) {
  const std::string &name = g_names[f];
  g_log += name + "\n";
  if (!grid.x || !grid.y || !grid.z || !block.x) return fail(INVALID);
  if (name.find("k_span_widths") != std::string::npos) {
    uint64_t *out = *(uint64_t **)args[4];
    const uint32_t n = *(uint32_t *)args[0];
    for (uint32_t k = 0; k < 10; ++k) {
      const double w = g_spacing * (4u << k);
      if ((4u << k) < n) memcpy(out + k, &w, 8);
      else out[k] = ~0ull;
    }
  }
  if (g_hook) g_hook(name.c_str(), args);
  return 0;
}

int hipMalloc(void **p, size_t n) { return alloc(p, n); }
int hipFree(void *p) {
  free(p);
  return 0;
}
// page-locked host memory: allocations, and what a test registers
void fake_register(void *p, size_t n) { g_host[(char *)p] = n; }
int hipHostMalloc(void **p, size_t n, unsigned) {
  const int rc = alloc(p, n);
  if (!rc) fake_register(*p, n);
  return rc;
}
int hipHostFree(void *p) {
  g_host.erase((char *)p);
  return hipFree(p);
}
int hipMemGetAddressRange(void **base, size_t *size, void *p) {
  auto it = g_host.upper_bound((char *)p);
  if (it == g_host.begin() || (--it, (char *)p >= it->first + it->second)) return fail(INVALID);
  *base = it->first;
  *size = it->second;
  return 0;
}
struct Attributes {
  int type, device;
  void *device_pointer, *host_pointer;
};
int hipPointerGetAttributes(Attributes *a, void *p) {
  void *base;
  size_t size;
  if (hipMemGetAddressRange(&base, &size, p)) return INVALID;
  *a = {1 /* hipMemoryTypeHost */, 0, p, p};
  return 0;
}
int hipMemcpy(void *d, const void *s, size_t n, int) {
  if (n) memmove(d, s, n);
  return 0;
}
int hipMemcpyAsync(void *d, const void *s, size_t n, int k, void *) {
  return hipMemcpy(d, s, n, k);
}
int hipMemset(void *d, int v, size_t n) {
  if (n) memset(d, v, n);
  return 0;
}
int hipMemsetAsync(void *d, int v, size_t n, void *) { return hipMemset(d, v, n); }

int hipGetDeviceCount(int *n) {
  *n = 1;
  return 0;
}
int hipGetDevice(int *d) {
  *d = 0;
  return 0;
}
int hipSetDevice(int) { return 0; }
int hipDeviceGetAttribute(int *v, int, int) {
  *v = 65536;
  return 0;
}
int hipDeviceSynchronize() { return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  *n = 1;
  return 0;
}
int hipFuncSetAttribute(const void *, int, int) { return 0; }
int hipGetSymbolAddress(void **, const void *) { return fail(INVALID); }
int hipGetLastError() {
  const int e = g_last;
  g_last = 0;
  return e;
}
const char *hipGetErrorString(int e) { return e == OOM ? "out of memory" : "error"; }

static int token(void **p) {
  *p = &g_token;
  return 0;
}
int hipStreamCreate(void **s) { return token(s); }
int hipStreamCreateWithFlags(void **s, unsigned) { return token(s); }
int hipStreamDestroy(void *) { return 0; }
int hipStreamSynchronize(void *) { return 0; }
int hipStreamWaitEvent(void *, void *, unsigned) { return 0; }
int hipEventCreate(void **e) {
  *e = calloc(1, sizeof(int));  // whether it has been recorded
  return 0;
}
int hipEventCreateWithFlags(void **e, unsigned) { return hipEventCreate(e); }
int hipEventDestroy(void *e) {
  free(e);
  return 0;
}
int hipEventRecord(void *e, void *) {
  *(int *)e = 1;
  return 0;
}
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *a, void *) {
  if (!*(int *)a) return fail(INVALID);  // never recorded
  *ms = 1.f;
  return 0;
}

}  // extern "C"
