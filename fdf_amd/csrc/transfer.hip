// transfer.hip -- arrays of the caller's host memory to and from the device.
//
// The caller's arrays are ordinary memory in 64-bit types; the device's are
// 32- or 64-bit, cell-linear or packed.  A kernel converts a chunk of the
// array between the device and a slot of pinned host memory, over the link,
// and the host copies between the slot and the caller's array: no device
// buffer, no pass over the array on the host, and the link, the conversion
// and the host's copy of successive chunks overlap.  What bounds it is the
// link (57 GB/s each way with one large copy) and, on one thread, the host's
// copy (9 to 30 GB/s, the less where pages are touched for the first time),
// so that a large transfer's chunks are shared out to threads that live for
// the call.  In place of pageable copies and loops over the elements: 16.8M
// particles' positions and PIDs down 65.6 -> 12.7 ms (42 GB/s), 400,000
// particles up 2.4 -> 1.0 ms and down 4.3 -> 1.2, 10,000 down 0.17 -> 0.08.
#include "transfer.hpp"

#include <string.h>

#include <atomic>
#include <memory>
#include <mutex>
#include <new>
#include <thread>
#include <vector>

namespace picgpu {

// 1 MiB slots: the gap between two launches costs the link a tenth of a
// slot's time (kernels writing 1 MiB: 52 GB/s, 256 KiB 43, 128 KiB 35).  A
// small transfer fills its slots less, so that the host's copies overlap too,
// but not below 512 KiB: an event and its wait take about 10 us.
constexpr size_t kSlotBytes = 1 << 20, kMinFill = 512 << 10;
// One thread more for every 2 MiB, up to 7: memory copies reach 30 GB/s on one
// thread, 81 on four, 124 on eight; starting 7 threads takes 0.1 ms.
constexpr size_t kBytesPerThread = 2 << 20;
// Small transfers: by the calling thread alone, through three slots.  A helper
// thread gains from 2 MiB down (positions of 2.4 MB: 125 -> 100 us) and costs up
// to 4 MiB up (2.4 MB of FP32 swarm: 122 -> 136 us, 3.6 MB 155 -> 167).
constexpr size_t kSmallDown = 2 << 20, kSmallUp = 4 << 20;
constexpr int kMaxThreads = 7;
// workgroups of a chunk's kernel: reads over the link lose where many
// wavefronts issue them (1 MiB: 32 workgroups 50 GB/s, 512 38), writes do not
constexpr int kDownBlocks = 128, kUpBlocks = 32;

// ---------------------------------------------------------------- kernels
// the two values out[e], out[e + 1] of a chunk as one 16-byte store
template <typename F>
__global__ __launch_bounds__(kBlock) void k_pack(int64_t e0, int64_t m, F f, unsigned long long *__restrict__ out) {
  for (int64_t q = 2 * ((int64_t)blockIdx.x * kBlock + threadIdx.x); q < m; q += 2 * (int64_t)gridDim.x * kBlock) {
    if (q + 1 < m) {
      ulonglong2 v;
      v.x = f(e0 + q);
      v.y = f(e0 + q + 1);
      *reinterpret_cast<ulonglong2 *>(out + q) = v;
    } else {
      out[q] = f(e0 + q);
    }
  }
}
__device__ __forceinline__ unsigned long long bits(double v) { return (unsigned long long)__double_as_longlong(v); }

struct PackCopy {
  const unsigned long long *src;
  __device__ __forceinline__ unsigned long long operator()(int64_t e) const { return src[e]; }
};
struct PackF32 {
  const float *src;
  __device__ __forceinline__ unsigned long long operator()(int64_t e) const { return bits((double)src[e]); }
};
struct PackI32 {
  const int32_t *src;
  __device__ __forceinline__ unsigned long long operator()(int64_t e) const { return (unsigned long long)(int64_t)src[e]; }
};
// component e % 3 of the cell of particle e / 3; -1 without a cell
struct PackCell {
  const int32_t *src;
  int IM, JM;
  __device__ __forceinline__ unsigned long long operator()(int64_t e) const {
    const int64_t p = e / 3;
    const int a = (int)(e - 3 * p);
    const int32_t c = src[p];
    if (c < 0) return (unsigned long long)(int64_t)-1;
    const int32_t r = c / IM;
    return (unsigned long long)(int64_t)(a == 0 ? c - r * IM : a == 1 ? r % JM : r / JM);
  }
};
// node slot e of a per-cell array: the cell (i,j,k) sits at node (i,j,k), the other slots hold 0
template <typename T>
struct PackNode {
  const T *src;
  int IM, JM, KM;
  __device__ __forceinline__ unsigned long long operator()(int64_t e) const {
    const int64_t r = e / (IM + 1);
    const int i = (int)(e - r * (IM + 1));
    const int64_t k = r / (JM + 1);
    const int j = (int)(r - k * (JM + 1));
    return i < IM && j < JM && k < KM ? bits((double)src[(k * JM + j) * IM + i]) : bits(0.0);
  }
};
template <typename R>
struct PackVolfrac {
  int dir;
  GridView g;
  const R *face;
  double vp;
  __device__ __forceinline__ unsigned long long operator()(int64_t f) const {
    return bits(face_volfrac<R>(dir, g, face, vp, f));
  }
};

template <typename F>
__global__ __launch_bounds__(kBlock) void k_unpack(int64_t e0, int64_t m, F f,
                                                   const unsigned long long *__restrict__ in) {
  for (int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x; q < m; q += (int64_t)gridDim.x * kBlock)
    f(e0 + q, in, q);
}
struct UnpackCopy {
  unsigned long long *dst;
  __device__ __forceinline__ void operator()(int64_t e, const unsigned long long *in, int64_t q) const { dst[e] = in[q]; }
};
struct UnpackF32 {
  float *dst;
  __device__ __forceinline__ void operator()(int64_t e, const unsigned long long *in, int64_t q) const {
    dst[e] = (float)__longlong_as_double((long long)in[q]);
  }
};
struct UnpackI32 {
  int32_t *dst;
  __device__ __forceinline__ void operator()(int64_t e, const unsigned long long *in, int64_t q) const {
    dst[e] = (int32_t)(int64_t)in[q];
  }
};
// packed cell of three indices, -1 outside the grid
struct UnpackCell {
  int32_t *dst;
  int IM, JM, KM;
  __device__ __forceinline__ void operator()(int64_t e, const unsigned long long *in, int64_t q) const {
    const int64_t i = (int64_t)in[3 * q], j = (int64_t)in[3 * q + 1], k = (int64_t)in[3 * q + 2];
    const bool ok = i >= 0 && j >= 0 && k >= 0 && i < IM && j < JM && k < KM;
    dst[e] = ok ? (int32_t)(i + (int64_t)IM * (j + (int64_t)JM * k)) : -1;
  }
};
template <typename R>
__global__ __launch_bounds__(kBlock) void k_fill_real(int64_t n, R v, R *__restrict__ out) {
  const int64_t q = (int64_t)blockIdx.x * kBlock + threadIdx.x;
  if (q < n) out[q] = v;
}

// times a chunk's launch from whichever thread of the transfer makes it
struct ChunkTimer {
  picgpu_ctx *c;
  std::unique_lock<std::mutex> lock;
  TimerRec rec;
  ChunkTimer(picgpu_ctx *ctx, const char *name) : c(ctx) {
    rec.a = rec.b = nullptr;
    if (!c->timing) return;
    lock = std::unique_lock<std::mutex>(c->timing_mu);
    c->pending.reserve(c->pending.size() + 1);
    timer_begin(c, name, rec);
  }
  ~ChunkTimer() { timer_end(c, rec); }
};

static int chunk_blocks(int64_t m, int per_thread, int most) {
  const int64_t b = (m + (int64_t)kBlock * per_thread - 1) / ((int64_t)kBlock * per_thread);
  return (int)(b < most ? b : most);
}

static hipError_t launch_pack(picgpu_ctx *c, const HostSeg &s, int64_t e0, int64_t m, void *slot) {
  auto go = [&](auto f) {
    ChunkTimer timer(c, s.kind == HostKind::Volfrac ? "face_volfrac" : "host_pack");
    hipLaunchKernelGGL(k_pack<decltype(f)>, dim3(chunk_blocks(m, 2, kDownBlocks)), dim3(kBlock), 0, c->stream, e0, m,
                       f, static_cast<unsigned long long *>(slot));
    return hipGetLastError();
  };
  const bool f32 = c->opt.precision == PICGPU_FP32;
  switch (s.kind) {
    case HostKind::Real:
      if (f32) return go(PackF32{static_cast<const float *>(s.dev)});
      return go(PackCopy{static_cast<const unsigned long long *>(s.dev)});
    case HostKind::Copy8: return go(PackCopy{static_cast<const unsigned long long *>(s.dev)});
    case HostKind::Int32: return go(PackI32{static_cast<const int32_t *>(s.dev)});
    case HostKind::Cell: return go(PackCell{static_cast<const int32_t *>(s.dev), c->IM, c->JM});
    case HostKind::NodeCount: return go(PackNode<int32_t>{static_cast<const int32_t *>(s.dev), c->IM, c->JM, c->KM});
    case HostKind::NodeReal:
      if (f32) return go(PackNode<float>{static_cast<const float *>(s.dev), c->IM, c->JM, c->KM});
      return go(PackNode<double>{static_cast<const double *>(s.dev), c->IM, c->JM, c->KM});
    case HostKind::Volfrac: {
      const GridView g{c->coor.as<double>(), c->IM, c->JM, c->KM};
      if (f32) return go(PackVolfrac<float>{s.dir, g, static_cast<const float *>(s.dev), c->particle_volume});
      return go(PackVolfrac<double>{s.dir, g, static_cast<const double *>(s.dev), c->particle_volume});
    }
  }
  return hipErrorInvalidValue;
}

static hipError_t launch_unpack(picgpu_ctx *c, const HostSeg &s, int64_t e0, int64_t m, const void *slot) {
  auto go = [&](auto f) {
    ChunkTimer timer(c, "host_unpack");
    hipLaunchKernelGGL(k_unpack<decltype(f)>, dim3(chunk_blocks(m, 1, kUpBlocks)), dim3(kBlock), 0, c->stream, e0, m,
                       f, static_cast<const unsigned long long *>(slot));
    return hipGetLastError();
  };
  switch (s.kind) {
    case HostKind::Real:
      if (c->opt.precision == PICGPU_FP32) return go(UnpackF32{static_cast<float *>(s.dev)});
      return go(UnpackCopy{static_cast<unsigned long long *>(s.dev)});
    case HostKind::Copy8: return go(UnpackCopy{static_cast<unsigned long long *>(s.dev)});
    case HostKind::Int32: return go(UnpackI32{static_cast<int32_t *>(s.dev)});
    case HostKind::Cell: return go(UnpackCell{static_cast<int32_t *>(s.dev), c->IM, c->JM, c->KM});
    default: return hipErrorInvalidValue;
  }
}

// ---------------------------------------------------------------- the ring
// The slots.  The host's first touch of pinned memory costs 0.38 ms a MiB (a
// fault a page), so the rings of transfers that have ended are kept for the
// next ones, at most kRingsKept of each size, until the last context is
// destroyed.  A small transfer has a ring of its own size: the runtime hands
// back an allocation below 2 MiB that it has seen before, already mapped, where
// 8 MiB are new each time that a program's only context is made again
// (20,000 particles, a context's first upload: 0.13 to 1.2 ms with the large
// ring, by whether they were, 0.12 with the small one; steady state 0.09 both).
// A transfer holds its ring alone; any device may use it.  The host rewrites a
// slot while later kernels are queued, and reads one while earlier ones run, so
// the memory is coherent by its own flag, whatever the environment asks of
// unflagged allocations (same time a transfer: 200,000 particles down 596 and
// 598 us, 2,000,000 up 6.11 and 6.11 ms).
struct RingSize {
  int slots;
  size_t slot_bytes;
};
constexpr RingSize kSmallRing{3, kMinFill}, kLargeRing{TransferEvents::kSlots, kSlotBytes};
constexpr int kRingsKept = 2;
static std::mutex g_rings_mu;
static void *g_rings[2][kRingsKept];  // small, large
static int g_ring_users;

void rings_open() {
  std::lock_guard<std::mutex> lock(g_rings_mu);
  ++g_ring_users;
}
void rings_close() {
  std::lock_guard<std::mutex> lock(g_rings_mu);
  if (--g_ring_users > 0) return;
  for (auto &size : g_rings)
    for (void *&r : size) {
      if (r) (void)hipHostFree(r);
      r = nullptr;
    }
}
static int take_ring(bool small, void **out) {
  {
    std::lock_guard<std::mutex> lock(g_rings_mu);
    for (void *&r : g_rings[small ? 0 : 1])
      if (r) {
        *out = r;
        r = nullptr;
        return PICGPU_OK;
      }
  }
  const RingSize &s = small ? kSmallRing : kLargeRing;
  if (hipHostMalloc(out, s.slot_bytes * s.slots, hipHostMallocPortable | hipHostMallocCoherent) == hipSuccess)
    return PICGPU_OK;
  (void)hipGetLastError();
  *out = nullptr;
  return PICGPU_E_NOMEM;
}
static void give_ring(bool small, void *ring) {
  {
    std::lock_guard<std::mutex> lock(g_rings_mu);
    for (void *&r : g_rings[small ? 0 : 1])
      if (!r) {
        r = ring;
        return;
      }
  }
  (void)hipHostFree(ring);
}

void TransferEvents::release() {
  for (hipEvent_t &e : ev) {
    if (e) (void)hipEventDestroy(e);
    e = nullptr;
  }
}

namespace {
// elements [e0, e0 + m) of an array, at byte `at` of their slot
struct Chunk {
  int seg;
  int64_t e0, m;
  size_t at;
};
// the chunks [first, end) that share a slot, so that many small arrays take one event
struct Group {
  size_t first, end;
};

// One transfer, shared by the calling thread and its helpers.  Group k goes
// through slot k % size.slots.
//  down: any thread may issue the next group's kernels (one thread at a time,
//        in order, into a slot whose last group was copied out); threads claim
//        issued groups, wait for the group's event and copy.
//  up:   threads claim groups in order, wait until the kernels of the slot's
//        last group have run, copy in, and launch.
// Every wait is for a group with a smaller number, which some thread has
// claimed or can issue, and ends on an error.
struct Transfer {
  picgpu_ctx *c;
  char *ring;
  RingSize size;
  const HostSeg *segs;
  const std::vector<Chunk> &chunks;
  const std::vector<Group> &groups;
  std::atomic<unsigned char> *done;  // down: copied out; up: kernel launched
  bool down;
  std::atomic<int64_t> issued{0}, claimed{0};
  std::atomic_flag issuing = ATOMIC_FLAG_INIT;
  std::atomic<int> err{0};

  char *slot(int64_t k) const { return ring + (size_t)(k % size.slots) * size.slot_bytes; }
  hipEvent_t event(int64_t k) const { return c->transfer.ev[k % size.slots]; }
  void copy(int64_t k) const {
    for (size_t q = groups[(size_t)k].first; q < groups[(size_t)k].end; ++q) {
      const Chunk &ch = chunks[q];
      const HostSeg &s = segs[ch.seg];
      char *h = static_cast<char *>(s.host) + (size_t)ch.e0 * s.stride;
      if (down)
        memcpy(h, slot(k) + ch.at, (size_t)ch.m * s.stride);
      else
        memcpy(slot(k) + ch.at, h, (size_t)ch.m * s.stride);
    }
  }
  bool launch(int64_t k) {
    for (size_t q = groups[(size_t)k].first; q < groups[(size_t)k].end; ++q) {
      const Chunk &ch = chunks[q];
      const HostSeg &s = segs[ch.seg];
      const int64_t w = (int64_t)(s.stride / 8);  // 8-byte values an element
      if (!ok(down ? launch_pack(c, s, ch.e0 * w, ch.m * w, slot(k) + ch.at)
                   : launch_unpack(c, s, ch.e0, ch.m, slot(k) + ch.at)))
        return false;
    }
    return ok(hipEventRecord(event(k), c->stream));
  }
  bool ok(hipError_t e) {
    if (e == hipSuccess) return true;
    int none = 0;
    err.compare_exchange_strong(none, (int)e);
    return false;
  }
  void issue() {
    if (issuing.test_and_set(std::memory_order_acquire)) return;
    const int64_t N = (int64_t)groups.size();
    for (int64_t k = issued.load(); k < N && !err.load(); ++k) {
      if (k >= size.slots && !done[k - size.slots].load(std::memory_order_acquire)) break;
      if (!launch(k)) break;
      issued.store(k + 1, std::memory_order_release);
    }
    issuing.clear(std::memory_order_release);
  }
  void run_down() {
    const int64_t N = (int64_t)groups.size();
    while (!err.load()) {
      issue();
      int64_t k = claimed.load();
      if (k >= N) return;
      if (k >= issued.load(std::memory_order_acquire) || !claimed.compare_exchange_strong(k, k + 1)) {
        std::this_thread::yield();
        continue;
      }
      if (!ok(hipEventSynchronize(event(k)))) return;
      copy(k);
      done[k].store(1, std::memory_order_release);
    }
  }
  void run_up() {
    const int64_t N = (int64_t)groups.size();
    while (!err.load()) {
      const int64_t k = claimed.fetch_add(1);
      if (k >= N) return;
      if (k >= size.slots) {
        while (!done[k - size.slots].load(std::memory_order_acquire)) {
          if (err.load()) return;
          std::this_thread::yield();
        }
        if (!ok(hipEventSynchronize(event(k)))) return;
      }
      copy(k);
      if (!launch(k)) return;
      done[k].store(1, std::memory_order_release);
    }
  }
  void run() {
    try {
      if (down)
        run_down();
      else
        run_up();
    } catch (...) {
      (void)ok(hipErrorOutOfMemory);
    }
  }
};
}  // namespace

static int move_host(picgpu_ctx *c, void *ring, bool small, const HostSeg *segs, int nsegs, size_t total, bool down) {
  size_t fill = total / kLargeRing.slots;
  fill = small || fill < kMinFill ? kMinFill : fill > kSlotBytes ? kSlotBytes : fill;
  std::vector<std::thread> helpers;
  try {
    std::vector<Chunk> chunks;
    std::vector<Group> groups;
    size_t used = fill;  // bytes of the last group's slot
    for (int s = 0; s < nsegs; ++s) {
      const size_t stride = segs[s].stride;
      for (int64_t e = 0; e < segs[s].n;) {
        if (used + stride > fill) {
          groups.push_back(Group{chunks.size(), chunks.size()});
          used = 0;
        }
        const int64_t room = (int64_t)((fill - used) / stride), m = segs[s].n - e < room ? segs[s].n - e : room;
        chunks.push_back(Chunk{s, e, m, used});
        groups.back().end = chunks.size();
        used = (used + (size_t)m * stride + 15) / 16 * 16;  // the kernels store 16 bytes
        e += m;
      }
    }
    std::unique_ptr<std::atomic<unsigned char>[]> done(new std::atomic<unsigned char>[groups.size()]);
    for (size_t k = 0; k < groups.size(); ++k) done[k].store(0);
    const RingSize size = small ? kSmallRing : kLargeRing;
    Transfer t{c, static_cast<char *>(ring), size, segs, chunks, groups, done.get(), down};
    if (down) t.issue();
    const size_t want = small ? 0 : total / kBytesPerThread;
    const int nth = want < (size_t)kMaxThreads ? (int)want : kMaxThreads;
    try {
      helpers.reserve((size_t)nth);
      for (int k = 0; k < nth; ++k)
        helpers.emplace_back([&t, c] {
          if (t.ok(hipSetDevice(c->device))) t.run();
        });
    } catch (...) {
      // fewer helpers: the calling thread and those that started do the work
    }
    t.run();
    for (std::thread &h : helpers) h.join();
    // a download has waited for every kernel's event
    const hipError_t e = down && !t.err.load() ? hipSuccess : hipStreamSynchronize(c->stream);
    const int te = t.err.load() ? t.err.load() : (int)e;
    if (te != hipSuccess) {
      set_error("host transfer failed: %s", hipGetErrorString((hipError_t)te));
      return PICGPU_E_HIP;
    }
  } catch (const std::bad_alloc &) {
    set_error("host transfer: out of host memory");
    return PICGPU_E_NOMEM;
  }
  return PICGPU_OK;
}

// Without pinned memory (a limit of the process or the machine): the kernels
// convert between the arrays and a slot of device memory, which the runtime
// copies from and to the caller's pageable arrays, a chunk after another.
static int move_pageable(picgpu_ctx *c, const HostSeg *segs, int nsegs, bool down) {
  DevBuf slot;
  PG_CHECK(slot.ensure(kSlotBytes));
  hipError_t err = hipSuccess;
  for (int s = 0; s < nsegs && err == hipSuccess; ++s) {
    const size_t stride = segs[s].stride;
    const int64_t w = (int64_t)(stride / 8), most = (int64_t)(kSlotBytes / stride);
    for (int64_t e = 0; e < segs[s].n && err == hipSuccess; e += most) {
      const int64_t m = segs[s].n - e < most ? segs[s].n - e : most;
      const size_t bytes = (size_t)m * stride;
      char *h = static_cast<char *>(segs[s].host) + (size_t)e * stride;
      if (down) {
        err = launch_pack(c, segs[s], e * w, m * w, slot.ptr);
        if (err == hipSuccess) err = hipMemcpyAsync(h, slot.ptr, bytes, hipMemcpyDeviceToHost, c->stream);
      } else {
        err = hipMemcpyAsync(slot.ptr, h, bytes, hipMemcpyHostToDevice, c->stream);
        if (err == hipSuccess) err = launch_unpack(c, segs[s], e, m, slot.ptr);
      }
      const hipError_t done = hipStreamSynchronize(c->stream);
      if (err == hipSuccess) err = done;
    }
  }
  slot.release();
  if (err != hipSuccess) {
    set_error("host transfer failed: %s", hipGetErrorString(err));
    return PICGPU_E_HIP;
  }
  return PICGPU_OK;
}

static int host_transfer(picgpu_ctx *c, const HostSeg *segs, int nsegs, bool down) {
  size_t total = 0;
  for (int s = 0; s < nsegs; ++s) total += (size_t)segs[s].n * segs[s].stride;
  if (total == 0) return PICGPU_OK;
  for (hipEvent_t &e : c->transfer.ev)
    if (!e) PG_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  const bool small = total < (down ? kSmallDown : kSmallUp);
  void *ring = nullptr;
  if (take_ring(small, &ring) != PICGPU_OK) return move_pageable(c, segs, nsegs, down);
  const int r = move_host(c, ring, small, segs, nsegs, total, down);
  give_ring(small, ring);
  return r;
}

int host_download(picgpu_ctx *c, const HostSeg *segs, int nsegs) { return host_transfer(c, segs, nsegs, true); }
int host_upload(picgpu_ctx *c, const HostSeg *segs, int nsegs) { return host_transfer(c, segs, nsegs, false); }

int fill_real(picgpu_ctx *c, void *dev, int64_t n, double v) {
  if (n <= 0) return PICGPU_OK;
  const dim3 grid((unsigned)((n + kBlock - 1) / kBlock));
  if (c->opt.precision == PICGPU_FP32)
    hipLaunchKernelGGL(k_fill_real<float>, grid, dim3(kBlock), 0, c->stream, n, (float)v, static_cast<float *>(dev));
  else
    hipLaunchKernelGGL(k_fill_real<double>, grid, dim3(kBlock), 0, c->stream, n, v, static_cast<double *>(dev));
  PG_HIP(hipGetLastError());
  return PICGPU_OK;
}

}  // namespace picgpu
