// hostio.hip -- bulk transfers between pageable host arrays and the device,
// and the device blocks that calls take and give back.
//
// A plain copy of a pageable array goes through the runtime's staging with
// one host thread that also takes the page faults of a fresh array: F2 of 4
// species on 20x25x35x72 (40 MB) took 4.0 ms to the host, 10 GB/s of the
// link's 57.  Here chunks go through a ring of pinned slots while several
// threads copy between the slots and the array.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

#include "ctx.h"

namespace {

using namespace ramgpu_host;

// Smaller arrays take the runtime's own copy.  A whole get_f2 by it and by the
// ring: 9 MB 0.53 -> 0.48 ms into pages that are there, 0.65 -> 0.61 into fresh
// ones, 40 MB 4.0 -> 1.7, 265 MB 25.9 -> 8.7.  A whole put_f2, where no pages
// are faulted in: 34 MB 1.06 -> 1.09, 36 MB 1.21 -> 1.13, 40 MB 1.46 -> 1.21,
// 100 MB 3.6 -> 2.6 (10 MB 0.33 -> 0.58).
constexpr size_t kPipeMinToHost = size_t(8) << 20, kPipeMinToDevice = size_t(34) << 20;
constexpr int kSlots = 8;
constexpr size_t kSlotBytes = size_t(4) << 20; // 32 MiB of pinned memory per process
constexpr int kMaxThreads = 6;
constexpr size_t kCacheMax = size_t(4) << 30;  // device bytes kept between calls, per process
constexpr unsigned long kPassedOver = 128;     // takes and gives (an adjoint makes about 30)

// The ring, one per process: a transfer takes it for its whole length; one
// that finds it taken uses the runtime's copy.  Its memory comes with the
// first large transfer and goes with the last context.
struct Pipe {
  std::mutex mu;
  char *mem = nullptr;
  hipEvent_t ev[kSlots] = {};
  int device = -1;

  void drop() {
    for (hipEvent_t &e : ev)
      if (e) {
        (void)hipEventDestroy(e);
        e = nullptr;
      }
    if (mem) (void)hipHostFree(mem);
    mem = nullptr;
    device = -1;
  }
  // with mu held and `dev` current: ready for transfers of that device
  bool ready(int dev) {
    if (mem && device == dev) return true;
    drop();
    if (hipHostMalloc((void **)&mem, kSlots * kSlotBytes, hipHostMallocPortable) != hipSuccess) {
      mem = nullptr;
      (void)hipGetLastError();
      return false;
    }
    for (hipEvent_t &e : ev)
      if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
        e = nullptr;
        (void)hipGetLastError();
        drop();
        return false;
      }
    device = dev;
    return true;
  }
};
Pipe g_pipe;
std::mutex g_live_mu;
int g_live = 0;  // contexts alive in the process

struct Block {
  int device;
  size_t bytes;
  void *p;
  unsigned long given;  // g_clock then
};
struct Taken {
  void *p;
  unsigned long when;
};
std::mutex g_cache_mu;
std::vector<Block> g_cache;  // in the order they were given back
std::vector<Taken> g_taken;  // the blocks that calls hold
size_t g_cached = 0;
unsigned long g_clock = 0;  // takes and gives so far

// One transfer through the ring (mu held).  Chunk i uses slot i mod kSlots.
struct Transfer {
  Pipe &pipe;
  int device;
  hipStream_t stream;
  char *host;
  char *dev;
  size_t bytes, chunk;
  int n;
  bool to_host;
  std::atomic<int> next{0}, issued{0}, err{0};
  std::vector<std::atomic<char>> done;

  Transfer(Pipe &p, int d, hipStream_t s, char *h, char *g, size_t b, size_t c, bool th)
      : pipe(p), device(d), stream(s), host(h), dev(g), bytes(b), chunk(c), n((int)((b + c - 1) / c)), to_host(th),
        done(n) {
    for (auto &x : done) x.store(0);
  }
  size_t len(int i) const { return std::min(chunk, bytes - (size_t)i * chunk); }
  char *slot(int i) const { return pipe.mem + (size_t)(i % kSlots) * kSlotBytes; }
  void check(hipError_t e) {
    if (e != hipSuccess) err.store((int)e);
  }
  // device to host: the calling thread issues the device copies of chunks
  // whose slots are free
  void issue() {
    for (int i = issued.load(); i < n && (i < kSlots || done[i - kSlots].load(std::memory_order_acquire)); ++i) {
      check(hipMemcpyAsync(slot(i), dev + (size_t)i * chunk, len(i), hipMemcpyDeviceToHost, stream));
      check(hipEventRecord(pipe.ev[i % kSlots], stream));
      issued.store(i + 1, std::memory_order_release);
    }
  }
  void work(bool issuer) {
    for (int i; (i = next.fetch_add(1)) < n;) {
      hipEvent_t e = pipe.ev[i % kSlots];
      if (to_host) {
        while (issued.load(std::memory_order_acquire) <= i) {
          if (issuer) issue();
          else std::this_thread::yield();
        }
        check(hipEventSynchronize(e));
        if (!err.load()) std::memcpy(host + (size_t)i * chunk, slot(i), len(i));
        done[i].store(1, std::memory_order_release);
        if (issuer) issue();
      } else {
        if (i >= kSlots) {  // the slot's previous chunk has left it
          while (!done[i - kSlots].load(std::memory_order_acquire)) std::this_thread::yield();
          check(hipEventSynchronize(e));
        }
        std::memcpy(slot(i), host + (size_t)i * chunk, len(i));
        check(hipMemcpyAsync(dev + (size_t)i * chunk, slot(i), len(i), hipMemcpyHostToDevice, stream));
        check(hipEventRecord(e, stream));
        done[i].store(1, std::memory_order_release);
      }
    }
    if (issuer && to_host)
      while (issued.load() < n) {
        issue();
        std::this_thread::yield();
      }
  }
  hipError_t run(int threads) {
    std::vector<std::thread> helpers;
    helpers.reserve(threads);
    if (to_host) issue();
    try {
      for (int t = 1; t < threads; ++t)
        helpers.emplace_back([this] {
          check(hipSetDevice(device));
          work(false);
        });
    } catch (const std::exception &) {  // no more threads, or no memory for one: those there, and this one, do it
    }
    work(true);
    for (std::thread &t : helpers) t.join();
    check(hipStreamSynchronize(stream));
    return (hipError_t)err.load();
  }
};

// Copy of `bytes` in stream order; dev is a device pointer.
int bulk_copy(int device, hipStream_t stream, void *host, void *dev, size_t bytes, bool to_host) {
  if (bytes >= (to_host ? kPipeMinToHost : kPipeMinToDevice)) {
    // asked for here only: the count is read from the system, 10 us
    const int cpus = (int)std::thread::hardware_concurrency();
    const int threads = std::min(kMaxThreads, std::max(1, cpus / 2));
    std::unique_lock<std::mutex> lk(g_pipe.mu, std::defer_lock);
    if (threads > 1 && lk.try_lock() && g_pipe.ready(device)) {
      // four chunks a thread, so that the last ones end together
      size_t chunk = bytes / ((size_t)threads * 4);
      chunk = std::min(kSlotBytes, std::max(size_t(512) << 10, chunk)) & ~size_t(4095);
      try {
        Transfer t(g_pipe, device, stream, (char *)host, (char *)dev, bytes, chunk, to_host);
        const hipError_t e = t.run(std::min(threads, t.n));
        if (e != hipSuccess) return fail(RAMGPU_EHIP, "transfer of %zu bytes: %s", bytes, hipGetErrorString(e));
        return RAMGPU_OK;
      } catch (const std::bad_alloc &) {  // the transfer's own tables, before its first copy
      }
    }
  }
  if (!to_host) {
    HIP_TRY(hipMemcpyAsync(dev, host, bytes, hipMemcpyHostToDevice, stream));
    return RAMGPU_OK;
  }
  HIP_TRY(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, stream));
  HIP_TRY(hipStreamSynchronize(stream));
  return RAMGPU_OK;
}

// with g_cache_mu held: kept block i out of the list
Block unkeep_locked(size_t i) {
  const Block b = g_cache[i];
  g_cache.erase(g_cache.begin() + i);
  g_cached -= b.bytes;
  return b;
}

// with g_cache_mu held
void trim_locked(int device) {
  for (size_t i = 0; i < g_cache.size();) {
    if (device < 0 || g_cache[i].device == device)
      (void)hipFree(unkeep_locked(i).p);
    else
      ++i;
  }
}

}  // namespace

namespace ramgpu_host {

int copy_to_host(int device, hipStream_t stream, void *host, const void *dev, size_t bytes) {
  return bulk_copy(device, stream, host, const_cast<void *>(dev), bytes, true);
}

int copy_to_device(int device, hipStream_t stream, void *dev, const void *host, size_t bytes) {
  return bulk_copy(device, stream, const_cast<void *>(host), dev, bytes, false);
}

bool dev_malloc(int device, void **p, size_t bytes) {
  if (hipMalloc(p, bytes) == hipSuccess) return true;
  (void)hipGetLastError();
  {
    std::lock_guard<std::mutex> lk(g_cache_mu);
    trim_locked(device);
  }
  if (hipMalloc(p, bytes) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

bool dev_take(int device, void **p, size_t bytes) {
  auto taken = [&] {  // with g_cache_mu held
    try {
      g_taken.push_back({*p, ++g_clock});
    } catch (const std::bad_alloc &) {  // given back, it finds room or goes
    }
    return true;
  };
  {
    std::lock_guard<std::mutex> lk(g_cache_mu);
    for (size_t i = 0; i < g_cache.size(); ++i)
      if (g_cache[i].device == device && g_cache[i].bytes == bytes) {
        *p = unkeep_locked(i).p;
        return taken();
      }
  }
  if (!dev_malloc(device, p, bytes)) return false;
  std::lock_guard<std::mutex> lk(g_cache_mu);
  return taken();
}

void dev_give(int device, void *p, size_t bytes) {
  std::lock_guard<std::mutex> lk(g_cache_mu);
  unsigned long when = 0;
  ++g_clock;
  for (size_t i = g_taken.size(); i-- > 0;)
    if (g_taken[i].p == p) {
      when = g_taken[i].when;
      g_taken.erase(g_taken.begin() + i);
      break;
    }
  // Blocks that several calls have passed over make room, the oldest first: a
  // size that is no longer asked for leaves in time, while the blocks of one
  // call, or of two that take turns, do not displace one another (an adjoint of
  // more than 4 GiB 30.6 ms, 38.6 with its own oldest blocks freed)
  if (bytes <= kCacheMax)
    while (g_cached + bytes > kCacheMax && !g_cache.empty() && g_cache[0].given + kPassedOver < when)
      (void)hipFree(unkeep_locked(0).p);
  if (g_cached + bytes <= kCacheMax) {
    try {
      g_cache.push_back({device, bytes, p, g_clock});
      g_cached += bytes;
      return;
    } catch (const std::bad_alloc &) {
    }
  }
  (void)hipFree(p);
}

size_t dev_cached(int device) {
  std::lock_guard<std::mutex> lk(g_cache_mu);
  size_t n = 0;
  for (const Block &b : g_cache)
    if (b.device == device) n += b.bytes;
  return n;
}

void context_opened() {
  std::lock_guard<std::mutex> lk(g_live_mu);
  ++g_live;
}

void context_closed() {
  std::lock_guard<std::mutex> lk(g_live_mu);
  if (--g_live > 0) return;
  {
    std::lock_guard<std::mutex> lc(g_cache_mu);
    trim_locked(-1);
  }
  std::lock_guard<std::mutex> lp(g_pipe.mu);
  g_pipe.drop();
}

}  // namespace ramgpu_host
