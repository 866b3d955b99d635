// bnz_xfer.hpp -- state arrays between the caller's host memory and the
// device (bnz_xfer.hip).
#pragma once
#include <hip/hip_runtime.h>

#include <mutex>

namespace bnz {

// `rows` rows of `len` doubles: back to back at host, `pitch` apart at dev.
struct Seg {
  double *dev;
  double *host;
  long pitch, rows, len;
  __host__ __device__ long total() const { return rows * len; }
};

// The host side of one context or batch: a pinned buffer of 1 MB, or 16 MB from
// the first larger transfer on, allocated when it is first needed and held until
// the object goes.  Any thread may call.
//   The runtime's own path for pageable memory costs 10 to 30 us a copy (a batch
// box is twelve), and one thread takes the pages of a new array's first touch (512
// MB down to new pages: 65 ms, 8 GB/s; 29 ms to old ones).  Here a small transfer,
// all its rows, is one launch that reads or writes the pinned buffer over the bus,
// and a large one is cut into chunks that a few host threads take, whose copies
// and page faults overlap the bus (57 GB/s; 8 threads copy 512 MB to new pages in
// 7 ms).
class HostLink {
 public:
  ~HostLink();
  // Copy n segments (at most 2) to the device or from it, in stream order; the
  // host memory is the caller's again on return, and down() has filled it.
  hipError_t up(int device, hipStream_t stream, const Seg *s, int n);
  hipError_t down(int device, hipStream_t stream, const Seg *s, int n);

 private:
  hipError_t move(int device, hipStream_t stream, const Seg *s, int n, bool to_dev);
  hipError_t direct(hipStream_t stream, const Seg *s, int n, bool to_dev);
  hipError_t reserve(hipStream_t stream, size_t bytes);
  std::mutex mu_;
  char *pin_ = nullptr;
  size_t cap_ = 0;    // its size
  size_t used_ = 0;   // bytes of it that uploads in flight may still read
  hipEvent_t ev_[8] = {};
  bool no_pin_ = false;
};

}  // namespace bnz
