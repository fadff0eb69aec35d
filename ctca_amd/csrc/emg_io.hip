// emg_io.hip -- host transfers of the entry points.  The caller's arrays are
// pageable memory, often fresh pages that fault on first touch: a plain copy
// reached 17 GB/s into warm pages and 9.5 GB/s into new ones, where the link
// does 56.  A transfer goes through a ring of pinned slots instead (at most
// kIoSlots x kIoSlot = 8 MB per context): kernels fill or drain the slots in
// chunks, addressing them directly, so there is no device staging, while up to
// kIoThreads host threads copy between slots and the caller's array.  50 MB of
// fields into new pages 5.3 -> 2.0 ms, 113 MB of records up 6.6 -> 2.7 ms and
// down 11.4 -> 3.5; 14 MB of eb up 0.44 -> 0.39 ms, 216 MB 7.4 -> 5.3, without the
// device staging of the same size that a plain copy and a splitting kernel need.
// (Uploads that are stored as they come stay plain copies.)  Chunk i is handled by thread i mod T,
// and with T dividing kIoSlots the chunk that reuses a slot belongs to the
// thread that used it last, so the threads share nothing.
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>

#include "emg_internal.h"

namespace emg {
namespace {

constexpr size_t kIoSlot = size_t(1) << 20;
constexpr size_t kIoOne = size_t(256) << 10;   // up to here one chunk
constexpr size_t kIoMany = size_t(4) << 20;    // from here several threads
constexpr int kIoThreads = 4;
static_assert(kIoSlots % kIoThreads == 0, "a slot's chunks belong to one thread");

__global__ __launch_bounds__(kBlock) void k_copy8(const unsigned long long *src, int64_t n,
                                                  unsigned long long *dst) {
  const int64_t o = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (o < n) dst[o] = src[o];
}

__global__ void k_flag(const int *dflag, int *hflag) {
  hflag[0] = dflag[0];
  hflag[1] = dflag[1];
}

// Pinned memory is slow to get (0.3 ms per MB), so a context that ends leaves
// its slots to the next one on its device: at most kPoolRings of them, given
// back when the last context of the process ends.
constexpr size_t kPoolRings = 4;
struct Ring {
  int device;
  char *pin;
  size_t bytes;
};
std::mutex g_mu;
int g_contexts = 0;
Ring g_pool[kPoolRings];
size_t g_pooled = 0;

// slots of at least `need` bytes for a device, from the pool or new
char *ring_get(int device, size_t need, size_t &bytes) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    for (size_t k = 0; k < g_pooled; k++)
      if (g_pool[k].device == device && g_pool[k].bytes >= need) {
        char *p = g_pool[k].pin;
        bytes = g_pool[k].bytes;
        g_pool[k] = g_pool[--g_pooled];
        return p;
      }
  }
  char *p = nullptr;
  if (hipHostMalloc((void **)&p, need, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  bytes = need;
  return p;
}

void ring_put(int device, char *pin, size_t bytes) {
  {
    std::lock_guard<std::mutex> lock(g_mu);
    if (g_contexts > 0 && g_pooled < kPoolRings) {
      g_pool[g_pooled++] = Ring{device, pin, bytes};
      return;
    }
  }
  (void)hipHostFree(pin);
}

struct Plan {
  size_t bytes, chunk;
  int n, threads;
};

int threads_for(size_t bytes) {
  const unsigned hc = std::thread::hardware_concurrency();
  return bytes >= kIoMany && (hc == 0 || hc >= (unsigned)kIoThreads) ? kIoThreads : 1;
}

Plan plan_of(size_t bytes, size_t unit) {
  Plan p;
  p.bytes = bytes;
  size_t chunk = bytes;
  if (bytes > kIoOne) {
    chunk = (bytes + kIoSlots - 1) / kIoSlots;
    if (chunk < kIoOne / 2) chunk = kIoOne / 2;
    if (chunk > kIoSlot) chunk = kIoSlot;
    chunk -= chunk % unit;
  }
  p.chunk = chunk;
  p.n = (int)((bytes + chunk - 1) / chunk);
  p.threads = threads_for(bytes);
  return p;
}

// The ring's slots, of at least `chunk` bytes each.  An upload still in the
// stream reads them: the host waits for it before it writes them again (what
// the GPU writes comes after it anyway).
int ring(emg_ctx *c, const Plan &p, bool host_writes) {
  HostIo &io = c->io;
  const int slots = p.n < kIoSlots ? p.n : kIoSlots;
  const size_t stride = (p.chunk + 255) / 256 * 256, need = stride * slots;
  if (io.pending && (host_writes || need > io.bytes)) {
    const int rc = hip_check(hipStreamSynchronize(c->stream), "stream synchronize");
    if (rc) return rc;
    io.pending = false;
  }
  if (need > io.bytes) {
    if (io.pin) ring_put(c->device, io.pin, io.bytes);
    io.bytes = 0;
    io.pin = ring_get(c->device, need, io.bytes);
    if (!io.pin) return set_error(EMG_ERR_NOMEM, "pinned transfer slots");
  }
  for (int k = 0; k < (p.n > 1 ? slots : 0); k++)
    if (!io.ev[k] && hipEventCreateWithFlags(&io.ev[k], hipEventDisableTiming) != hipSuccess) {
      io.ev[k] = nullptr;
      return set_error(EMG_ERR_HIP, "transfer event");
    }
  io.stride = stride;
  return EMG_OK;
}

// f(t) for t = 0..threads - 1, each on its own thread; what cannot get a thread
// runs on the caller's.  Returns the first error; f does not throw.
template <class F>
int on_threads(emg_ctx *c, int threads, F f) {
  if (threads == 1) return f(0);
  std::atomic<int> rc{EMG_OK};
  auto one = [&](int t) {
    int r = EMG_OK;
    if (t != 0 && hipSetDevice(c->device) != hipSuccess) r = EMG_ERR_HIP;
    if (!r) r = f(t);
    int ok = EMG_OK;
    if (r) rc.compare_exchange_strong(ok, r);
  };
  std::thread th[kIoThreads];
  int started = 1;
  try {
    for (; started < threads; started++) th[started] = std::thread(one, started);
  } catch (...) {  // no more threads: the rest below
  }
  one(0);
  for (int t = started; t < threads; t++) one(t);
  for (int t = 1; t < started; t++) th[t].join();
  const int r = rc.load();
  // a worker's message stayed with its thread
  return r ? set_error(r, "host transfer failed") : EMG_OK;
}

}  // namespace

void io_open(emg_ctx *c) {
  std::lock_guard<std::mutex> lock(g_mu);
  c->io.open = true;
  g_contexts++;
}

// (the context's stream is idle)
void io_close(emg_ctx *c) {
  HostIo &io = c->io;
  for (hipEvent_t &e : io.ev)
    if (e) (void)hipEventDestroy(e);
  Ring old[kPoolRings];
  size_t n = 0;
  if (io.open) {
    std::lock_guard<std::mutex> lock(g_mu);
    if (--g_contexts == 0) {
      n = g_pooled;
      for (size_t k = 0; k < n; k++) old[k] = g_pool[k];
      g_pooled = 0;
    }
  }
  for (size_t k = 0; k < n; k++) (void)hipHostFree(old[k].pin);
  if (io.pin) ring_put(c->device, io.pin, io.bytes);
  io = HostIo{};
}

int read_flags(emg_ctx *c) {
  hipLaunchKernelGGL(k_flag, dim3(1), dim3(1), 0, c->stream, c->dflag, c->hflag);
  const int rc = hip_check(hipStreamSynchronize(c->stream), "stream synchronize");
  return rc ? rc : flags_error(c);
}

int io_read(emg_ctx *c, void *user, size_t bytes, size_t unit, const IoFn &fill, bool flags) {
  if (bytes == 0) return flags ? read_flags(c) : EMG_OK;
  const Plan p = plan_of(bytes, unit);
  int rc = ring(c, p, false);
  if (rc) return rc;
  HostIo &io = c->io;
  const int slots = p.n < kIoSlots ? p.n : kIoSlots;
  auto enqueue = [&](int i) {
    const size_t off = (size_t)i * p.chunk, len = i == p.n - 1 ? bytes - off : p.chunk;
    const int s = i % slots;
    int r = fill(off, len, io.pin + s * io.stride);
    if (!r && p.n > 1) r = hip_check(hipEventRecord(io.ev[s], c->stream), "transfer event");
    return r;
  };
  if (flags) hipLaunchKernelGGL(k_flag, dim3(1), dim3(1), 0, c->stream, c->dflag, c->hflag);
  for (int i = 0; i < slots && !rc; i++) rc = enqueue(i);
  // device-side errors are reported before anything reaches the caller's array
  if (!rc)
    rc = p.n == 1 ? hip_check(hipStreamSynchronize(c->stream), "stream synchronize")
                  : hip_check(hipEventSynchronize(io.ev[0]), "stream synchronize");
  if (!rc && flags) rc = flags_error(c);
  if (rc) {
    (void)hipStreamSynchronize(c->stream);
    return rc;
  }
  if (p.n == 1) {
    std::memcpy(user, io.pin, bytes);
    return EMG_OK;
  }
  rc = on_threads(c, p.threads, [&](int t) {
    int r = EMG_OK;
    for (int i = t; i < p.n && !r; i += p.threads) {
      const size_t off = (size_t)i * p.chunk, len = i == p.n - 1 ? bytes - off : p.chunk;
      r = hip_check(hipEventSynchronize(io.ev[i % slots]), "transfer");
      if (r) break;
      std::memcpy(static_cast<char *>(user) + off, io.pin + (i % slots) * io.stride, len);
      if (i + slots < p.n) r = enqueue(i + slots);
    }
    return r;
  });
  if (rc) (void)hipStreamSynchronize(c->stream);
  return rc;
}

int io_read_array(emg_ctx *c, void *user, const void *dev, size_t bytes, bool flags) {
  const IoFn fill = [c, dev](size_t off, size_t len, void *slot) {
    const int64_t n = (int64_t)(len / 8);
    hipLaunchKernelGGL(k_copy8, dim3((unsigned)((n + kBlock - 1) / kBlock)), dim3(kBlock), 0,
                       c->stream, (const unsigned long long *)((const char *)dev + off), n,
                       (unsigned long long *)slot);
    return hip_check(hipGetLastError(), "read-out");
  };
  return io_read(c, user, bytes, 8, fill, flags);
}

int io_ranges(emg_ctx *c, int64_t n, size_t bytes,
              const std::function<void(int64_t, int64_t)> &f) {
  const int threads = threads_for(bytes * (size_t)n);
  return on_threads(c, threads, [&](int t) {
    f(n * t / threads, n * (t + 1) / threads);
    return EMG_OK;
  });
}

int io_write(emg_ctx *c, const void *user, size_t bytes, size_t unit, const IoFn &use,
             const IoCopy &copy) {
  if (bytes == 0) return EMG_OK;
  const Plan p = plan_of(bytes, unit);
  int rc = ring(c, p, true);
  if (rc) return rc;
  HostIo &io = c->io;
  const int slots = p.n < kIoSlots ? p.n : kIoSlots;
  rc = on_threads(c, p.threads, [&](int t) {
    int r = EMG_OK;
    for (int i = t; i < p.n && !r; i += p.threads) {
      const size_t off = (size_t)i * p.chunk, len = i == p.n - 1 ? bytes - off : p.chunk;
      const int s = i % slots;
      if (i >= slots) r = hip_check(hipEventSynchronize(io.ev[s]), "transfer");
      if (r) break;
      char *slot = io.pin + s * io.stride;
      size_t got = len;
      if (copy)
        got = copy(off, len, slot);
      else
        std::memcpy(slot, static_cast<const char *>(user) + off, len);
      if (got > 0) r = use(off, got, slot);
      if (!r && i + slots < p.n)
        r = hip_check(hipEventRecord(io.ev[s], c->stream), "transfer event");
    }
    return r;
  });
  if (rc)
    (void)hipStreamSynchronize(c->stream);
  else
    io.pending = true;  // the slots are in use until the stream gets there
  return rc;
}

}  // namespace emg
