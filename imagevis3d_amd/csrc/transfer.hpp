// transfer.hpp -- large copies between the caller's memory and the device.
//
// The runtime stages a copy from or to pageable memory through its own
// pinned buffers with one thread: 28 GB/s to the device and 17 GB/s back on
// this machine, where pinned copies reach 57 GB/s both ways.  Here worker
// threads move the pieces between the caller's memory and a pinned buffer
// each while other pieces are on the link.  The workers serve the whole
// device (paging needs them too): a transfer takes them once the work queued
// before it is done and gives them up, after the pieces at hand, to anyone
// who waits for them; while they are busy, pieces go the runtime's way.
#pragma once
#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include <condition_variable>
#include <mutex>

namespace tvk {

struct CopyPiece {
  void* dst;
  const void* src;
  size_t bytes;
};

// One stream's staging buffers: kSlots pinned buffers of kChunk bytes (16
// MiB of the device's CPU budget that nobody else uses), made when the
// owner's large copies have come to kWorth bytes and given back with the
// owner, or when the budget is needed for anything else.  Used by one thread
// at a time, like the renderer it belongs to.
class HostPipe {
 public:
  static constexpr size_t kChunk = 2u << 20;
  static constexpr int kSlots = 8;
  // Smaller copies take the runtime's path: waking the workers costs more.
  static constexpr size_t kLeast = 4u << 20;
  // Making and freeing the buffers takes about 1.2 ms, which the pinned path
  // wins back over 35 (device to host) to 85 MB: a renderer that loads 4 MiB
  // and goes took 1.55 ms for both against 0.48 without the buffers.
  static constexpr size_t kWorth = 64u << 20;

  ~HostPipe() { Release(); }
  // Neither copy throws.  Upload queues the copy on `stream`; `src` stays as
  // it is until the stream has passed it.
  hipError_t Upload(int device, void* dst, const void* src, size_t bytes, hipStream_t stream);
  // Copies device memory out after the work queued on `stream`; the data is
  // in host memory when it returns.
  hipError_t Download(int device, const CopyPiece* pieces, size_t n, hipStream_t stream);
  void Release();

 private:
  struct Loan;
  bool begin(int device, size_t bytes);  // the buffers are there, and ours until end()
  void end();
  void give(bool wait);
  void drop();  // frees the buffers; mu_ held
  static void give_back(int device, bool wait);
  int device_ = -1;
  std::mutex mu_;  // busy_ and, while it is false, all below
  std::condition_variable idle_;
  bool busy_ = false;  // a transfer is using the buffers
  size_t moved_ = 0;   // large copies made without the buffers
  void* buf_[kSlots] = {};
  hipEvent_t ev_[kSlots] = {};
};

// Host-to-host copy on the device's worker threads (large blocks).
void parallel_memcpy(int device, void* dst, const void* src, size_t bytes);

}  // namespace tvk
