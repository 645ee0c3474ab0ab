// Per-cell and per-vertex arrays to the caller's memory in the reference's
// numbering (gfx950).  Included by cc_solver.hip and nc_solver.hip.
//
// The rows lie in storage order on the device.  A kernel gathers them in the
// reference's order straight into pinned host memory, where they arrive at
// the link's rate (64 MB in 1.2 ms), and the host copies them on into the
// caller's array.  Up to 4 MB that is one launch and one copy: 960 KB take
// 42 us, 4 MB 134 us into memory in use (a device copy to the array itself
// 55 and 235 us, and the permutation in a host loop came on top).  Larger
// arrays are mostly new memory, whose page faults are the larger part of the
// copy: there threads copy chunk by chunk while the next chunks arrive, and
// share the faults.  Two million rows of four doubles (64 MB) took 24 ms as a
// device copy with the host loop after it; with one, two, four and eight
// threads the whole takes 4.9, 3.0, 1.9 and 1.75 ms where the array is in
// huge pages, 13.5, 7.2, 5.1 and 3.3 ms where it is not.  Below 4 MB a
// thread's start (17 us) is more than it saves.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <memory>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "helper_threads.h"
#include "ufx_internal.h"

namespace ufx {

// Row i of dst is row map[i] of src.  W 4: half a row (16 bytes) a thread.
template <int W>
static __global__ __launch_bounds__(256) void k_gather_rows(const double* src, const int* map, size_t i0,
                                                     size_t n, double* dst) {
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (W == 4) {
    if (t >= 2 * n) return;
    const double2* s = reinterpret_cast<const double2*>(src);
    reinterpret_cast<double2*>(dst)[t] = s[2 * (size_t)map[i0 + t / 2] + (t & 1)];
  } else {
    if (t >= n) return;
    dst[t] = src[map[i0 + t]];
  }
}

constexpr size_t RB_RING = (size_t)16 << 20;     // pinned bytes of a context at most
constexpr size_t RB_MIN = (size_t)64 << 10;      // and at least
constexpr size_t RB_SINGLE = (size_t)4 << 20;    // one launch, one copy
constexpr size_t RB_CHUNK_MIN = (size_t)256 << 10, RB_CHUNK_MAX = (size_t)1 << 20;
constexpr int RB_SLOTS = (int)(RB_RING / RB_CHUNK_MIN);
constexpr size_t RB_SHARE = (size_t)2 << 20;     // bytes a thread, eight threads at most
constexpr int RB_THREADS = 8;

// A context's pinned memory.  Reserved when the context is made (the
// allocation takes 50 to 130 us); a read reserves it where that failed.
struct Readback {
  char* ring = nullptr;
  size_t cap = 0;
  hipEvent_t ev[RB_SLOTS] = {};

  void release() {
    if (ring) (void)hipHostFree(ring);
    ring = nullptr;
    cap = 0;
    for (hipEvent_t& e : ev) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
  }
  // At least 64 KB; as much of `bytes`, up to the ring's size, as there is.
  hipError_t reserve(size_t bytes) {
    size_t want = std::min(RB_RING, (std::max(bytes, RB_MIN) + RB_MIN - 1) / RB_MIN * RB_MIN);
    if (cap >= want) return hipSuccess;
    if (ring) (void)hipHostFree(ring);
    ring = nullptr;
    cap = 0;
    hipError_t e = hipSuccess;
    for (;; want = std::max(RB_MIN, want / 2 / RB_MIN * RB_MIN)) {
      e = hipHostMalloc((void**)&ring, want, hipHostMallocDefault);
      if (e == hipSuccess) break;
      (void)hipGetLastError();
      ring = nullptr;
      if (want == RB_MIN) return e;
    }
    cap = want;
    for (size_t i = 0; i < cap; i += 4096) ring[i] = 0;  // (mapped before the first read)
    return hipSuccess;
  }
};

// The context's device made current, the caller's put back at the end.
struct DeviceGuard {
  int was = -1;
  explicit DeviceGuard(int device) {
    if (hipGetDevice(&was) != hipSuccess || was == device || hipSetDevice(device) != hipSuccess)
      was = -1;
  }
  ~DeviceGuard() {
    if (was >= 0) (void)hipSetDevice(was);
  }
};

inline int read_failed(hipError_t e) {
  (void)hipGetLastError();
  set_error(std::string("read-back: ") + hipGetErrorString(e));
  return UFX_ERR_HIP;
}

// Rows map[0] .. map[n - 1] of src (hmap: the map on the host, a permutation of
// 0 .. n - 1) to dst.
template <int W>
static int read_rows(Readback& rb, int device, hipStream_t stream, const double* src, const int* map,
              const std::vector<int>& hmap, size_t n, double* dst) {
  constexpr size_t ROW = W * sizeof(double);
  const size_t bytes = n * ROW;
  if (n == 0) return UFX_OK;
  const DeviceGuard guard(device);
  if (rb.reserve(bytes) != hipSuccess) {
    // no pinned memory to be had: through the runtime's own, permuted here
    std::unique_ptr<double[]> t(new (std::nothrow) double[n * W]);
    if (!t) {
      set_error("read-back: out of host memory");
      return UFX_ERR_HIP;
    }
    hipError_t e = hipMemcpyAsync(t.get(), src, bytes, hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return read_failed(e);
    for (size_t i = 0; i < n; ++i) std::memcpy(dst + i * W, &t[(size_t)hmap[i] * W], ROW);
    return UFX_OK;
  }
  auto gather = [&](size_t i0, size_t m, char* to) {
    const size_t th = W == 4 ? 2 * m : m;
    k_gather_rows<W><<<(unsigned)((th + 255) / 256), 256, 0, stream>>>(src, map, i0, m,
                                                                       (double*)to);
    return hipGetLastError();
  };
  if (bytes <= RB_SINGLE && bytes <= rb.cap) {
    hipError_t e = gather(0, n, rb.ring);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return read_failed(e);
    std::memcpy(dst, rb.ring, bytes);
    return UFX_OK;
  }
  const size_t chunk =
      std::min(rb.cap, std::clamp(bytes / 16 / ROW * ROW, RB_CHUNK_MIN, RB_CHUNK_MAX)) / ROW * ROW;
  const int slots = (int)std::min<size_t>(RB_SLOTS, rb.cap / chunk);
  const size_t nch = (bytes + chunk - 1) / chunk;
  for (int i = 0; i < slots; ++i)
    if (!rb.ev[i])
      if (hipError_t e = hipEventCreateWithFlags(&rb.ev[i], hipEventDisableTiming))
        return read_failed(e);
  std::unique_ptr<std::atomic<char>[]> done(new (std::nothrow) std::atomic<char>[nch]);
  if (!done) {
    set_error("read-back: out of host memory");
    return UFX_ERR_HIP;
  }
  for (size_t c = 0; c < nch; ++c) done[c].store(0, std::memory_order_relaxed);
  std::atomic<size_t> issued{0}, next{0};
  std::atomic<int> bad{hipSuccess};
  // copies one issued chunk that no thread has taken; false if there is none
  auto copy_one = [&] {
    size_t c = next.load(std::memory_order_relaxed);
    do {
      if (c >= issued.load(std::memory_order_acquire)) return false;
    } while (!next.compare_exchange_weak(c, c + 1));
    const int sl = (int)(c % slots);
    if (hipError_t e = hipEventSynchronize(rb.ev[sl])) bad.store(e);
    else std::memcpy((char*)dst + c * chunk, rb.ring + sl * chunk, std::min(chunk, bytes - c * chunk));
    done[c].store(1, std::memory_order_release);
    return true;
  };
  auto help = [&] {
    if (hipError_t e = hipSetDevice(device)) { bad.store(e); return; }
    while (bad.load() == hipSuccess && next.load(std::memory_order_relaxed) < nch)
      if (!copy_one()) std::this_thread::yield();
  };
  std::thread th[RB_THREADS - 1];
  const int most = (int)std::min<size_t>(
      {RB_THREADS, bytes / RB_SHARE, std::max(1u, std::thread::hardware_concurrency())});
  // (the ones that start, and this thread, do it)
  const int nth = start_threads(th, most - 1, help);
  for (size_t c = 0; c < nch && bad.load() == hipSuccess; ++c) {
    // the slot's last chunk copied out
    while (c >= (size_t)slots && !done[c - slots].load(std::memory_order_acquire))
      if (!copy_one()) std::this_thread::yield();
    const size_t i0 = c * (chunk / ROW);
    hipError_t e = gather(i0, std::min(chunk / ROW, n - i0), rb.ring + (c % slots) * chunk);
    if (e == hipSuccess) e = hipEventRecord(rb.ev[c % slots], stream);
    if (e != hipSuccess) { bad.store(e); break; }
    issued.store(c + 1, std::memory_order_release);
  }
  while (bad.load() == hipSuccess && copy_one()) {
  }
  for (int i = 0; i < nth; ++i) th[i].join();
  // (after an error the stream may still write to the pinned memory)
  if (bad.load() != hipSuccess) {
    (void)hipStreamSynchronize(stream);
    return read_failed((hipError_t)bad.load());
  }
  return UFX_OK;
}

}  // namespace ufx
