// Runs hostio.hip's host code without a device: the HIP calls that it makes
// are stand-ins on host memory.  Arguments: the check to run; see
// test_hostio_host.py.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <new>
#include <vector>

#include "ctx.h"

static std::atomic<long> g_news_left{-1};  // allocations that still succeed (< 0: all)
static std::atomic<long> g_mallocs{0}, g_frees{0};
static std::atomic<size_t> g_malloc_bytes{0};

static void *counted(size_t n) {
  if (g_news_left.load() >= 0 && g_news_left.fetch_sub(1) <= 0) {
    g_news_left.store(0);
    throw std::bad_alloc();
  }
  if (void *p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void *operator new(size_t n) { return counted(n); }
void *operator new[](size_t n) { return counted(n); }
void operator delete(void *p) noexcept { std::free(p); }
void operator delete[](void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
void operator delete[](void *p, size_t) noexcept { std::free(p); }

extern "C" {
hipError_t hipMalloc(void **p, size_t n) {
  ++g_mallocs;
  g_malloc_bytes += n;
  *p = std::malloc(1);
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  ++g_frees;
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  *p = std::malloc(n);
  return hipSuccess;
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  *e = (hipEvent_t)std::malloc(1);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::free(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stand-in"; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return hipSuccess;
}
}

namespace ramgpu_host {
int fail(int code, const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  std::vfprintf(stderr, fmt, ap);
  va_end(ap);
  return code;
}
}  // namespace ramgpu_host

using namespace ramgpu_host;

#define EXPECT(x)                                        \
  do {                                                   \
    if (!(x)) {                                          \
      std::printf("line %d: %s\n", __LINE__, #x);        \
      return 1;                                          \
    }                                                    \
  } while (0)

// every allocation of a transfer in turn fails, and all after it
static int no_memory() {
  const size_t n = (size_t(40) << 20) + 4097;
  std::vector<unsigned char> a(n), b(n);
  for (size_t i = 0; i < n; ++i) a[i] = (unsigned char)(i * 2654435761u >> 13);
  for (long left = 0; left < 24; ++left)
    for (int to_host = 0; to_host < 2; ++to_host) {
      std::memset(b.data(), 0, n);
      g_news_left.store(left);
      const int rc = to_host ? copy_to_host(0, nullptr, b.data(), a.data(), n) : copy_to_device(0, nullptr, b.data(), a.data(), n);
      g_news_left.store(-1);
      EXPECT(rc == RAMGPU_OK);
      EXPECT(std::memcmp(a.data(), b.data(), n) == 0);
    }
  return 0;
}

// kept blocks: those of sizes no longer asked for make room for the latest
// call's; of a call that holds more than is kept, as many as fit stay
static int kept_blocks() {
  const size_t MB = size_t(1) << 20;
  void *p[8], *q;
  for (int first : {0, 4})
    for (int call = 0; call < 60; ++call) {
      const long m = g_mallocs;
      for (int i = first; i < first + 4; ++i) EXPECT(dev_take(0, &p[i], (900 + i) * MB));
      EXPECT(call < 58 || (g_mallocs == m && dev_cached(0) == 0));
      for (int i = first; i < first + 4; ++i) dev_give(0, p[i], (900 + i) * MB);
      EXPECT(dev_cached(0) <= 4096 * MB);
    }
  EXPECT(dev_cached(0) == (904 + 905 + 906 + 907) * MB);
  const size_t big[6] = {2000, 900, 700, 450, 300, 200};  // 4550: the last ones find no room
  for (int call = 0; call < 60; ++call) {
    const size_t b = g_malloc_bytes;
    for (int i = 0; i < 6; ++i) EXPECT(dev_take(1, &p[i], big[i] * MB));
    EXPECT(call < 58 || g_malloc_bytes - b <= 500 * MB);
    for (int i = 0; i < 6; ++i) dev_give(1, p[i], big[i] * MB);
    EXPECT(dev_take(0, &q, 100 * MB));  // a call in between
    dev_give(0, q, 100 * MB);
    EXPECT(dev_cached(0) + dev_cached(1) <= 4096 * MB);
  }
  EXPECT(dev_take(0, &q, 5000 * MB));  // more than is ever kept: the others stay
  const size_t kept = dev_cached(1);
  dev_give(0, q, 5000 * MB);
  EXPECT(kept > 4000 * MB && dev_cached(1) == kept);
  EXPECT(dev_take(0, &q, 900 * MB));  // another device's block is not this one's
  EXPECT(dev_cached(1) == kept);
  dev_give(0, q, 900 * MB);
  context_opened();
  context_closed();
  EXPECT(dev_cached(0) == 0 && dev_cached(1) == 0 && g_mallocs == g_frees);
  return 0;
}

int main(int argc, char **argv) {
  if (argc > 1 && !std::strcmp(argv[1], "no_memory")) return no_memory();
  if (argc > 1 && !std::strcmp(argv[1], "kept_blocks")) return kept_blocks();
  return 2;
}
