// bnz_xfer.hip -- transfers between host arrays and device state (HostLink).
#include "bnz_xfer.hpp"

#include <algorithm>
#include <atomic>
#include <cstring>
#include <thread>

namespace bnz {
namespace {

// The large pinned buffer: one chunk per worker of a large transfer.  Chunks of
// 2 MB are 37 us of bus time each, against about 5 us between launches.
constexpr int WORKERS = 8;
constexpr size_t CHUNK = 2u << 20, CAP = WORKERS * CHUNK;
constexpr long CHUNK_LEN = CHUNK / sizeof(double);
// The small one: up to 1 MB the runtime hands out pinned memory in 15 to 70 us,
// beyond in 300 to 900, and the first touch of its pages takes 0.4 us a KB.
constexpr size_t SMALL = 1u << 20;
// Below this plain arrays go through the runtime: two arrays of 50 KB take it
// 30 us up and 50 down.
constexpr size_t DIRECT = 64u << 10;
// From here on threads pay (starting one is some 20 us; one thread copies to
// new pages at 10 GB/s, to old ones at 40).  Four uploads and downloads of new
// arrays, a process's first, by the runtime -> so: 1.2 MB 4.7 -> 2.4 ms, 4.2 MB
// 12.8 -> 6.9, 19 MB 20.3 -> 7.8; 1 MB 3.9 -> 1.7 (2.3 with the large buffer).
constexpr size_t THREADED = 2 * CHUNK;
constexpr int BLOCK = 256, MAX_BLOCKS = 256;

// Elements e0 .. e0 + m - 1 of the segments, counted through a and then b,
// between their device rows and stage.
template <bool UP>
__global__ __launch_bounds__(BLOCK) void k_rows(Seg a, Seg b, double *stage, long e0, long m) {
  const long na = a.total();
  for (long q = (long)blockIdx.x * BLOCK + threadIdx.x; q < m; q += (long)gridDim.x * BLOCK) {
    long e = e0 + q;
    const bool first = e < na;
    if (!first) e -= na;
    const long len = first ? a.len : b.len, pitch = first ? a.pitch : b.pitch;
    double *p = (first ? a.dev : b.dev) + (len == pitch ? e : e / len * pitch + e % len);
    if (UP)
      *p = stage[q];
    else
      stage[q] = *p;
  }
}

// The host side of elements e0 .. e0 + m - 1.
void host_part(const Seg *s, int n, char *stage, long e0, long m, bool to_dev) {
  for (int k = 0; k < n && m > 0; ++k) {
    const long t = s[k].total();
    if (e0 < t) {
      const long take = std::min(m, t - e0);
      if (to_dev)
        std::memcpy(stage, s[k].host + e0, take * sizeof(double));
      else
        std::memcpy(s[k].host + e0, stage, take * sizeof(double));
      stage += take * sizeof(double);
      m -= take;
      e0 = 0;
    } else {
      e0 -= t;
    }
  }
}

// The caller's thread on the device of the stream, and back.
struct OnDevice {
  int before = -1;
  explicit OnDevice(int device) {
    int now;
    if (hipGetDevice(&now) == hipSuccess && now != device && hipSetDevice(device) == hipSuccess)
      before = now;
  }
  ~OnDevice() {
    if (before >= 0) (void)hipSetDevice(before);
  }
};

hipError_t launch_rows(hipStream_t stream, const Seg *s, int n, char *stage, long e0, long m,
                       bool to_dev) {
  const Seg b = n > 1 ? s[1] : Seg{nullptr, nullptr, 1, 0, 1};
  const dim3 grid((unsigned)std::min<long>((m + BLOCK - 1) / BLOCK, MAX_BLOCKS));
  if (to_dev)
    hipLaunchKernelGGL(k_rows<true>, grid, dim3(BLOCK), 0, stream, s[0], b, (double *)stage, e0, m);
  else
    hipLaunchKernelGGL(k_rows<false>, grid, dim3(BLOCK), 0, stream, s[0], b, (double *)stage, e0,
                       m);
  return hipGetLastError();
}

}  // namespace

HostLink::~HostLink() {
  if (pin_) (void)hipHostFree(pin_);
  for (hipEvent_t e : ev_)
    if (e) (void)hipEventDestroy(e);
}

// A pinned buffer for a transfer of so many bytes; cap_ stays too small where
// there is no memory for one.
hipError_t HostLink::reserve(hipStream_t stream, size_t bytes) {
  if (no_pin_ || bytes <= cap_ || cap_ == CAP) return hipSuccess;
  const size_t cap = bytes > SMALL ? CAP : SMALL;
  if (pin_) {  // uploads in flight may still read the old one
    const hipError_t e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return e;
    (void)hipHostFree(pin_);
    pin_ = nullptr;
    cap_ = used_ = 0;
  }
  if (hipHostMalloc((void **)&pin_, cap, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    pin_ = nullptr;
  } else {
    cap_ = cap;
  }
  no_pin_ = pin_ == nullptr;
  return hipSuccess;
}

// Row by row through the runtime.  (A download as a blocking copy behind a
// wait: two arrays of 5 KB 27 us, as asynchronous copies 37.)
hipError_t HostLink::direct(hipStream_t stream, const Seg *s, int n, bool to_dev) {
  if (!to_dev) {
    const hipError_t e = hipStreamSynchronize(stream);
    if (e != hipSuccess) return e;
  }
  for (int k = 0; k < n; ++k)
    for (long r = 0; r < s[k].rows; ++r) {
      double *d = s[k].dev + r * s[k].pitch, *h = s[k].host + r * s[k].len;
      const size_t bytes = s[k].len * sizeof(double);
      const hipError_t e = to_dev
                               ? hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, stream)
                               : hipMemcpy(h, d, bytes, hipMemcpyDeviceToHost);
      if (e != hipSuccess) return e;
    }
  return to_dev ? hipStreamSynchronize(stream) : hipSuccess;
}

hipError_t HostLink::move(int device, hipStream_t stream, const Seg *s, int n, bool to_dev) {
  if (n < 1) return hipSuccess;
  std::lock_guard<std::mutex> lock(mu_);
  const OnDevice on(device);
  const long total = s[0].total() + (n > 1 ? s[1].total() : 0);
  const size_t bytes = total * sizeof(double);
  const bool plain = s[0].rows == 1 && (n < 2 || s[1].rows == 1);
  if (plain && bytes < DIRECT) return direct(stream, s, n, to_dev);
  hipError_t e0 = reserve(stream, bytes);
  if (e0 != hipSuccess) return e0;
  if (cap_ < std::min(bytes, CAP)) return direct(stream, s, n, to_dev);
  if (bytes < THREADED) {
    hipError_t e = hipSuccess;
    if (used_ + bytes > cap_) {
      if ((e = hipStreamSynchronize(stream)) != hipSuccess) return e;
      used_ = 0;
    }
    char *stage = pin_ + used_;
    if (to_dev) {
      host_part(s, n, stage, 0, total, true);
      used_ += (bytes + 255) / 256 * 256;
      return launch_rows(stream, s, n, stage, 0, total, true);
    }
    if ((e = launch_rows(stream, s, n, stage, 0, total, false)) != hipSuccess) return e;
    if ((e = hipStreamSynchronize(stream)) != hipSuccess) return e;
    used_ = 0;
    host_part(s, n, stage, 0, total, false);
    return hipSuccess;
  }
  // Large: each worker owns a chunk of the buffer and takes the next piece of
  // the arrays when it is free, so the workers need no word with each other.
  if ((e0 = hipStreamSynchronize(stream)) != hipSuccess) return e0;
  used_ = 0;
  for (hipEvent_t &e : ev_)
    if (!e && (e0 = hipEventCreateWithFlags(&e, hipEventDisableTiming)) != hipSuccess) return e0;
  const long pieces = (total + CHUNK_LEN - 1) / CHUNK_LEN;
  std::atomic<long> next{0};
  std::atomic<int> error{hipSuccess};
  const auto work = [&](int w) {
    hipError_t e = hipSetDevice(device);
    char *stage = pin_ + w * CHUNK;
    long c;
    bool pending = false;
    while (e == hipSuccess && error.load() == hipSuccess && (c = next.fetch_add(1)) < pieces) {
      const long at = c * CHUNK_LEN, m = std::min(CHUNK_LEN, total - at);
      if (to_dev) {
        if (pending && (e = hipEventSynchronize(ev_[w])) != hipSuccess) break;
        host_part(s, n, stage, at, m, true);
      }
      if ((e = launch_rows(stream, s, n, stage, at, m, to_dev)) != hipSuccess) break;
      if ((e = hipEventRecord(ev_[w], stream)) != hipSuccess) break;
      pending = true;
      if (!to_dev) {
        if ((e = hipEventSynchronize(ev_[w])) != hipSuccess) break;
        host_part(s, n, stage, at, m, false);
      }
    }
    if (e != hipSuccess) error.store(e);
  };
  std::thread pool[WORKERS];
  const int workers = (int)std::min<long>(WORKERS, pieces);
  for (int w = 1; w < workers; ++w) {
    try {
      pool[w] = std::thread(work, w);
    } catch (...) {
      break;  // no more threads or memory: the others take the pieces
    }
  }
  work(0);
  for (std::thread &t : pool)
    if (t.joinable()) t.join();
  const hipError_t done = hipStreamSynchronize(stream);
  return error.load() != hipSuccess ? (hipError_t)error.load() : done;
}

hipError_t HostLink::up(int device, hipStream_t stream, const Seg *s, int n) {
  return move(device, stream, s, n, true);
}

hipError_t HostLink::down(int device, hipStream_t stream, const Seg *s, int n) {
  return move(device, stream, s, n, false);
}

}  // namespace bnz
