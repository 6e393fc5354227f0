// hostio.hip -- transfers between the caller's raw arrays and the device.
//
// The arrays are ordinary (pageable) host memory.  Copied by the runtime they
// reach 28 GB/s to the device and 17 GB/s back on this host, against 57 GB/s
// for pinned memory: its staging copy runs on one thread.  Here a transfer is
// cut into chunks of sites; several threads copy a chunk between the caller's
// array and a ring of pinned buffers while the neighbouring chunks are on the
// bus, and the layout conversion of a chunk runs as soon as it has arrived.
// Measured: a 191 MB field (24^4 links, FP64) in 6.8 -> 4.0 ms to the device,
// 11 -> 3.9 ms back; the four link arrays of 24^3x32 (1.02 GB, once instead of
// the long ones twice) 55 -> 23 ms; an 8^4 vector 50 -> 26 us in, 57 -> 25 us
// out.  That call on the links with other settings: the copy engine instead of
// the copy kernel 31 ms (41 with 4 MB chunks), 1024 blocks 38 ms, 4 / 12 / 16
// threads the same.
#include "hostio.h"
#include "copy_pool.h"

#include <sched.h>

#include <algorithm>
#include <cstring>
#include <mutex>

namespace qphix {

namespace {

constexpr size_t HOST_THREADED = (size_t)2 << 20;  // smaller transfers are copied by the caller alone
constexpr int HOST_THREADS = 8;
// Larger transfers cross the bus by a copy kernel of this many blocks (the copy
// engine waits for the compute queue around every chunk).
constexpr unsigned COPY_BLOCKS = 256;

// Copies n bytes (a multiple of 16) between device memory and a pinned buffer.
__global__ void __launch_bounds__(256) k_copy_host(uint4 *d, const uint4 *s, unsigned n16) {
  for (unsigned i = blockIdx.x * 256u + threadIdx.x; i < n16; i += gridDim.x * 256u) d[i] = s[i];
}
void queue_copy(char *d, const char *s, size_t n, hipStream_t stream) {
  const unsigned n16 = (unsigned)(n / 16);
  hipLaunchKernelGGL(k_copy_host, dim3(std::min((n16 + 255) / 256, COPY_BLOCKS)), dim3(256), 0, stream, reinterpret_cast<uint4 *>(d),
                     reinterpret_cast<const uint4 *>(s), n16);
  HIP_CHECK(hipGetLastError());
}

// One transfer at a time holds the ring; calls from several threads take turns.
// Recursive: an error during a transfer may end the process (fail()), and an exit
// handler that finalizes the library gives the ring back in the same thread.
struct Ring {
  std::recursive_mutex m;
  char *pinned = nullptr;
  hipEvent_t ev[HOST_BUFS] = {};
  CopyPool *pool = nullptr;
};
Ring &ring() {
  // never destroyed: its threads may be asleep when the process exits
  static Ring *r = new Ring;
  return *r;
}

// Pinned buffers on the first transfer; false without them (the runtime copies then).
bool ring_ready(Ring &r, bool threaded) {
  if (!r.pinned) {
    if (hipHostMalloc((void **)&r.pinned, HOST_CHUNK * HOST_BUFS, hipHostMallocDefault) != hipSuccess) {
      r.pinned = nullptr;
      (void)hipGetLastError();
      return false;
    }
    for (auto &e : r.ev) HIP_CHECK(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  if (threaded && !r.pool) {
    cpu_set_t set;
    const int cpus = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
    r.pool = new CopyPool(std::max(0, std::min(HOST_THREADS, cpus) - 1));
  }
  return true;
}

// Memory the CPU should not copy itself (pinned or device memory handed over as
// a raw array): the runtime copies it directly.
bool plain_host(const void *p) {
  hipPointerAttribute_t at{};
  if (hipPointerGetAttributes(&at, p) != hipSuccess) {
    (void)hipGetLastError();
    return true;
  }
  return at.type == hipMemoryTypeUnregistered;
}

// The chunk of every array inside a buffer of `p.chunk` sites.
void split(char *base, const HostArray *a, int na, const HostPlan &p, char **d) {
  for (int k = 0; k < na; ++k) {
    d[k] = base;
    base += a[k].bytes * p.chunk;
  }
}

struct Transfer {
  Ring &r;
  std::unique_lock<std::recursive_mutex> lock;
  HostPlan p;
  const HostArray *a;
  int na;
  bool staged[4], any = false, threaded;

  Transfer(const HostArray *a_, int na_, size_t half, int halves) : r(ring()), lock(r.m), a(a_), na(na_) {
    size_t per = 0;
    for (int k = 0; k < na; ++k) per += a[k].bytes;
    p = host_plan(per, half, halves);
    threaded = per * half * halves > HOST_THREADED;
    for (int k = 0; k < na; ++k) any |= staged[k] = plain_host(a[k].p);
    if (any && !ring_ready(r, threaded)) {  // no pinned memory: the runtime copies
      any = false;
      for (int k = 0; k < na; ++k) staged[k] = false;
    }
    p.direct = p.direct && any;
    for (int k = 0; k < na; ++k) p.direct = p.direct && staged[k];
    threaded = threaded && any;
    if (threaded) r.pool->open();
  }
  ~Transfer() {
    if (threaded) r.pool->close();
  }
  void copy(char *d, const char *s, size_t n) {
    if (threaded) r.pool->copy(d, s, n);
    else std::memcpy(d, s, n);
  }
};

} // namespace

void host_to_device(const HostArray *a, int na, size_t half, int halves, char *stage, const HostUse &use) {
  if (half == 0 || halves == 0) return;
  Transfer t(a, na, half, halves);
  hipStream_t s = ctx().stream;
  for (size_t c = 0; c < t.p.chunks; ++c) {
    const int b = (int)(c % t.p.nbuf);
    const size_t first = t.p.first(c), n = t.p.count(c);
    char *dev[4], *pin[4] = {};
    split(stage + t.p.per_site * t.p.chunk * b, a, na, t.p, dev);
    if (t.any) {
      split(t.r.pinned + HOST_CHUNK * b, a, na, t.p, pin);
      if (c >= (size_t)t.p.nbuf) HIP_CHECK(hipEventSynchronize(t.r.ev[b]));
    }
    for (int k = 0; k < na; ++k) {
      const char *src = a[k].p + first * a[k].bytes;
      if (t.staged[k]) t.copy(pin[k], src, n * a[k].bytes);
      if (t.p.direct) continue;
      if (t.staged[k]) queue_copy(dev[k], pin[k], n * a[k].bytes, s);
      else HIP_CHECK(hipMemcpyAsync(dev[k], src, n * a[k].bytes, hipMemcpyHostToDevice, s));
    }
    // the pinned buffer is free once it has been read: by the copy, or by use()
    if (t.any && !t.p.direct) HIP_CHECK(hipEventRecord(t.r.ev[b], s));
    use(t.p.direct ? pin : dev, first, n);
    if (t.p.direct) HIP_CHECK(hipEventRecord(t.r.ev[b], s));
  }
  HIP_CHECK(hipStreamSynchronize(s));
}

void device_to_host(const HostArray *a, int na, size_t half, int halves, char *stage, const HostUse &fill) {
  if (half == 0 || halves == 0) return;
  Transfer t(a, na, half, halves);
  hipStream_t s = ctx().stream;
  const size_t nc = t.p.chunks, nb = (size_t)t.p.nbuf;
  for (size_t c = 0; c < nc + nb; ++c) {
    if (c >= nb && t.any) {  // chunk c - nb to the caller's arrays
      const size_t o = c - nb;
      char *pin[4];
      split(t.r.pinned + HOST_CHUNK * (o % nb), a, na, t.p, pin);
      HIP_CHECK(hipEventSynchronize(t.r.ev[o % nb]));
      for (int k = 0; k < na; ++k)
        if (t.staged[k]) t.copy(a[k].p + t.p.first(o) * a[k].bytes, pin[k], t.p.count(o) * a[k].bytes);
    }
    if (c < nc) {
      const int b = (int)(c % nb);
      const size_t first = t.p.first(c), n = t.p.count(c);
      char *dev[4], *pin[4] = {};
      split(stage + t.p.per_site * t.p.chunk * b, a, na, t.p, dev);
      if (t.any) split(t.r.pinned + HOST_CHUNK * b, a, na, t.p, pin);
      fill(t.p.direct ? pin : dev, first, n);
      for (int k = 0; k < na && !t.p.direct; ++k) {
        if (t.staged[k]) queue_copy(pin[k], dev[k], n * a[k].bytes, s);
        else
          HIP_CHECK(hipMemcpyAsync(a[k].p + first * a[k].bytes, dev[k], n * a[k].bytes, hipMemcpyDeviceToHost, s));
      }
      if (t.any) HIP_CHECK(hipEventRecord(t.r.ev[b], s));
    }
  }
  HIP_CHECK(hipStreamSynchronize(s));
}

void host_io_release() {
  Ring &r = ring();
  std::lock_guard<std::recursive_mutex> l(r.m);
  delete r.pool;
  r.pool = nullptr;
  if (r.pinned) {
    HIP_CHECK(hipHostFree(r.pinned));
    for (auto &e : r.ev) HIP_CHECK(hipEventDestroy(e));
  }
  r.pinned = nullptr;
}

} // namespace qphix
