// A host stand-in for the part of the HIP runtime that bnz_xfer.hip uses, for
// tests of its control flow: device memory is host memory, and what is put on
// the one stream runs when somebody waits for it, not before.
#pragma once
#include <cstddef>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>

#define __host__
#define __device__
#define __global__
#define __launch_bounds__(...)

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;
struct dim3 {
  unsigned x;
  explicit dim3(unsigned n = 1) : x(n) {}
};
typedef struct FakeStream *hipStream_t;
typedef struct FakeEvent *hipEvent_t;
struct FakeStream {
  std::mutex mu;
  std::deque<std::function<void()>> queue;
  long done = 0, issued = 0;
  long put(std::function<void()> f) {
    std::lock_guard<std::mutex> l(mu);
    queue.push_back(std::move(f));
    return ++issued;
  }
  void wait(long upto) {
    std::lock_guard<std::mutex> l(mu);
    while (done < upto) {
      queue.front()();
      queue.pop_front();
      ++done;
    }
  }
};
struct FakeEvent {
  FakeStream *s = nullptr;
  long at = 0;
};

// what the test sets and reads
struct FakeHip {
  size_t pin_limit = ~size_t(0);  // larger pinned buffers are refused
  size_t pinned = 0, pins = 0;
  std::mutex mu;
  long copies = 0, launches = 0;
};
inline FakeHip fake;

inline thread_local dim3 blockIdx(0), threadIdx(0), gridDim(1);

inline hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
inline hipError_t hipSetDevice(int) { return hipSuccess; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (n > fake.pin_limit) return hipErrorOutOfMemory;
  fake.pinned = n;
  ++fake.pins;
  *p = std::malloc(n);
  return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
  std::free(p);
  fake.pinned = 0;
  return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
  return *e = new FakeEvent, hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  e->s = s;
  e->at = s->put([] {});
  return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e) {
  if (e->s) e->s->wait(e->at);
  return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
  long all;
  {
    std::lock_guard<std::mutex> l(s->mu);
    all = s->issued;
  }
  s->wait(all);
  return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t st) {
  {
    std::lock_guard<std::mutex> l(fake.mu);
    ++fake.copies;
  }
  st->put([=] { std::memcpy(d, s, n); });
  return hipSuccess;
}
inline hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  ++fake.copies;
  std::memcpy(d, s, n);  // (a blocking copy does not wait for a non-blocking stream)
  return hipSuccess;
}
template <class... A>
void fake_launch(void (*kernel)(A...), dim3 grid, dim3 block, hipStream_t s, A... args) {
  {
    std::lock_guard<std::mutex> l(fake.mu);
    ++fake.launches;
  }
  s->put([=] {
    gridDim = grid;
    for (unsigned b = 0; b < grid.x; ++b)
      for (unsigned t = 0; t < block.x; ++t) {
        blockIdx = dim3(b);
        threadIdx = dim3(t);
        kernel(args...);
      }
  });
}
#define hipLaunchKernelGGL(k, grid, block, lds, stream, ...) \
  fake_launch(k, grid, block, stream, __VA_ARGS__)
