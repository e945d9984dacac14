// transfer.cpp -- see transfer.hpp.
#include "transfer.hpp"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <vector>

#include "memman.hpp"

namespace tvk {
namespace {

// Memory the runtime can copy from or to directly (pinned or managed).
bool pinned(const void* p) {
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();  // ordinary memory: not an error of the caller's
    return false;
  }
  return a.type == hipMemoryTypeHost || a.type == hipMemoryTypeDevice || a.type == hipMemoryTypeManaged;
}

}  // namespace

bool HostPipe::ready(int device, size_t bytes) {
  if (buf_[0]) return device_ == device;
  if (tried_) return false;  // no memory for the buffers: the runtime's path
  if ((moved_ += bytes) < kWorth) return false;
  tried_ = true;
  MemMan& mm = MemMan::ForDevice(device);
  if (!mm.ReserveCPU(kSlots * kChunk)) return false;
  device_ = device;
  bool ok = true;
  for (int i = 0; i < kSlots && ok; ++i)
    ok = hipHostMalloc(&buf_[i], kChunk, hipHostMallocDefault) == hipSuccess &&
         hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming) == hipSuccess;
  if (!ok) {
    (void)hipGetLastError();
    Release();
    tried_ = true;
  }
  return ok;
}

void HostPipe::Release() {
  moved_ = 0;
  if (device_ < 0) return;
  for (int i = 0; i < kSlots; ++i) {
    if (ev_[i]) {
      (void)hipEventSynchronize(ev_[i]);  // its last copy may still read the buffer
      (void)hipEventDestroy(ev_[i]);
    }
    if (buf_[i]) (void)hipHostFree(buf_[i]);
    ev_[i] = nullptr;
    buf_[i] = nullptr;
  }
  MemMan::ForDevice(device_).ReleaseCPU(kSlots * kChunk);
  device_ = -1;
  tried_ = false;
}

hipError_t HostPipe::Upload(int device, void* dst, const void* src, size_t bytes, hipStream_t stream) {
  if (bytes >= kLeast && !pinned(src) && ready(device, bytes)) {
    const size_t n = (bytes + kChunk - 1) / kChunk;
    std::atomic<int> err{hipSuccess};
    const bool done = MemMan::ForDevice(device).TryParallelFor((size_t)kSlots, kSlots, [&](size_t t) {
      hipError_t e = hipSetDevice(device);
      for (size_t c = t; c < n && e == hipSuccess && err == hipSuccess; c += kSlots) {
        const size_t off = c * kChunk, len = std::min(kChunk, bytes - off);
        e = hipEventSynchronize(ev_[t]);  // the buffer's last copy (an event never recorded is done)
        if (e != hipSuccess) break;
        memcpy(buf_[t], (const char*)src + off, len);
        e = hipMemcpyAsync((char*)dst + off, buf_[t], len, hipMemcpyHostToDevice, stream);
        if (e == hipSuccess) e = hipEventRecord(ev_[t], stream);
      }
      if (e != hipSuccess) err = (int)e;
    });
    if (done) return (hipError_t)err.load();
  }
  return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream);
}

hipError_t HostPipe::Download(int device, const CopyPiece* pieces, size_t n, hipStream_t stream) {
  size_t total = 0;
  bool direct = false;
  for (size_t i = 0; i < n; ++i) {
    total += pieces[i].bytes;
    direct = direct || pinned(pieces[i].dst);
  }
  if (total >= kLeast && !direct && ready(device, total)) {
    std::vector<CopyPiece> cut;
    for (size_t i = 0; i < n; ++i)
      for (size_t off = 0; off < pieces[i].bytes; off += kChunk)
        cut.push_back(CopyPiece{(char*)pieces[i].dst + off, (const char*)pieces[i].src + off,
                                std::min(kChunk, pieces[i].bytes - off)});
    std::atomic<int> err{hipSuccess};
    const bool done = MemMan::ForDevice(device).TryParallelFor((size_t)kSlots, kSlots, [&](size_t t) {
      hipError_t e = hipSetDevice(device);
      for (size_t c = t; c < cut.size() && e == hipSuccess && err == hipSuccess; c += kSlots) {
        e = hipMemcpyAsync(buf_[t], cut[c].src, cut[c].bytes, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipEventRecord(ev_[t], stream);
        if (e == hipSuccess) e = hipEventSynchronize(ev_[t]);
        if (e == hipSuccess) memcpy(cut[c].dst, buf_[t], cut[c].bytes);
      }
      if (e != hipSuccess) err = (int)e;
    });
    if (done) return (hipError_t)err.load();
  }
  for (size_t i = 0; i < n; ++i)
    if (hipError_t e = hipMemcpyAsync(pieces[i].dst, pieces[i].src, pieces[i].bytes, hipMemcpyDeviceToHost, stream))
      return e;
  return hipStreamSynchronize(stream);
}

void parallel_memcpy(int device, void* dst, const void* src, size_t bytes) {
  constexpr size_t kPart = 1u << 20;
  const size_t n = (bytes + kPart - 1) / kPart;
  if (bytes < HostPipe::kLeast || !MemMan::ForDevice(device).TryParallelFor(n, HostPipe::kSlots, [&](size_t i) {
        const size_t off = i * kPart;
        memcpy((char*)dst + off, (const char*)src + off, std::min(kPart, bytes - off));
      }))
    memcpy(dst, src, bytes);
}

}  // namespace tvk
