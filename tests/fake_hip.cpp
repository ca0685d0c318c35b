// A HIP runtime of two devices in host memory, preloaded to run the library's
// host code where no GPU is: copies are done at once, launches do nothing.  It
// counts uses of a stream or event by a thread whose current device is another,
// and fails operator new on request.  Memory is taken only where it is touched,
// copies of 1 GB and more are left out, and launches of 2^32 work-items and more in
// a dimension are refused, as the real runtime does.
#include <sys/mman.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <atomic>
#include <new>

namespace {
struct Handle {
  int device;
};
struct Dim {
  uint32_t x, y, z;
};
thread_local int g_device = 0, g_fail_new = 0, g_error = 0;
thread_local Dim g_grid, g_block;
thread_local size_t g_shared;
thread_local void *g_stream;
std::atomic<int> g_cross{0}, g_foreign{0};

int use(void *h) {
  if (h && static_cast<Handle *>(h)->device != g_device) ++g_cross;
  return 0;
}
int make(void **h) {
  if (g_device != 0) ++g_foreign;
  if (!(*h = malloc(sizeof(Handle)))) return 2;
  static_cast<Handle *>(*h)->device = g_device;
  return 0;
}
int drop(void *h) {
  free(h);
  return 0;
}
int get(void **p, size_t n) {
  *p = mmap(nullptr, n + 4096, PROT_READ | PROT_WRITE,
            MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (*p == MAP_FAILED) return 2;
  *static_cast<size_t *>(*p) = n + 4096;  // the mapping's length, a page below
  *p = static_cast<char *>(*p) + 4096;
  return 0;
}
int put(void *p) {
  if (!p) return 0;
  void *base = static_cast<char *>(p) - 4096;
  return munmap(base, *static_cast<size_t *>(base));
}
void copy(void *d, const void *s, size_t n) {
  if (n < size_t(1) << 30) memcpy(d, s, n);
}
}  // namespace

void *operator new(size_t n) {
  if (g_fail_new && --g_fail_new == 0) throw std::bad_alloc();
  if (void *p = malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void operator delete(void *p) noexcept { free(p); }
void operator delete(void *p, size_t) noexcept { free(p); }

extern "C" {
int fake_cross() { return g_cross; }      // uses from another device
int fake_foreign() { return g_foreign; }  // streams and events made on device 1
void fake_fail_new(int k) { g_fail_new = k; }  // the k-th of this thread from here (0: none)

int hipGetDeviceCount(int *n) { return *n = 2, 0; }
int hipGetDevice(int *d) { return *d = g_device, 0; }
int hipSetDevice(int d) { return g_device = d, 0; }
int hipDeviceGetAttribute(int *v, int, int) { return *v = 256, 0; }
int hipDeviceSynchronize() { return 0; }
int hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int, size_t) {
  return *n = 4, 0;
}
int hipGetLastError() {
  const int e = g_error;
  g_error = 0;
  return e;
}
const char *hipGetErrorString(int) { return "fake"; }
int hipMalloc(void **p, size_t n) { return get(p, n); }
int hipFree(void *p) { return put(p); }
int hipHostMalloc(void **p, size_t n, unsigned) { return get(p, n); }
int hipHostFree(void *p) { return put(p); }
int hipStreamCreateWithFlags(void **s, unsigned) { return make(s); }
int hipStreamDestroy(void *s) { return drop(s); }
int hipStreamSynchronize(void *) { return 0; }
int hipStreamWaitEvent(void *s, void *, unsigned) { return use(s); }
int hipEventCreate(void **e) { return make(e); }
int hipEventCreateWithFlags(void **e, unsigned) { return make(e); }
int hipEventDestroy(void *e) { return drop(e); }
int hipEventRecord(void *e, void *s) { return use(e), use(s); }
int hipEventSynchronize(void *) { return 0; }
int hipEventElapsedTime(float *ms, void *, void *) { return *ms = 1.0f, 0; }
int hipMemcpy(void *d, const void *s, size_t n, int) { return copy(d, s, n), 0; }
int hipMemcpyAsync(void *d, const void *s, size_t n, int, void *stream) {
  copy(d, s, n);
  return use(stream);
}
int hipMemset(void *d, int v, size_t n) { return memset(d, v, n), 0; }
int hipMemsetAsync(void *d, int v, size_t n, void *stream) {
  memset(d, v, n);
  return use(stream);
}
int hipLaunchKernel(const void *, Dim grid, Dim block, void **, size_t, void *stream) {
  g_error = 0;
  const uint64_t limit = uint64_t(1) << 32;
  if (uint64_t(grid.x) * block.x >= limit || uint64_t(grid.y) * block.y >= limit ||
      uint64_t(grid.z) * block.z >= limit)
    return g_error = 9;  // hipErrorInvalidConfiguration
  return use(stream);
}
int __hipPushCallConfiguration(Dim grid, Dim block, size_t shared, void *stream) {
  g_grid = grid;
  g_block = block;
  g_shared = shared;
  g_stream = stream;
  return 0;
}
int __hipPopCallConfiguration(Dim *grid, Dim *block, size_t *shared, void **stream) {
  *grid = g_grid;
  *block = g_block;
  *shared = g_shared;
  *stream = g_stream;
  return 0;
}
void **__hipRegisterFatBinary(const void *) { return static_cast<void **>(calloc(1, 64)); }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *,
                           void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
}
