// transfer.cpp -- see transfer.hpp.
#include "transfer.hpp"

#include <string.h>

#include <algorithm>
#include <atomic>
#include <functional>
#include <map>
#include <new>
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

// Runs piece(c, slot) for pieces [0, n) on the workers: slot t has the pieces
// t, t + kSlots, .. from next[t] on, one after the other, and stops early
// when someone else needs the workers.  False, and nothing done, when they
// are busy.
template <typename F>
bool pooled(int device, size_t n, size_t (&next)[HostPipe::kSlots], const F& piece, hipError_t* err) {
  MemMan& mm = MemMan::ForDevice(device);
  std::atomic<int> first{hipSuccess};
  auto slot = [&](size_t t) {
    hipError_t e = hipSetDevice(device);
    for (; next[t] < n && e == hipSuccess && first == hipSuccess && !mm.WorkersWanted(); next[t] += HostPipe::kSlots)
      e = piece(next[t], t);
    if (e != hipSuccess) first = (int)e;
  };
  // by reference: a std::function of it needs no memory
  const bool ran = mm.TryParallelFor((size_t)HostPipe::kSlots, HostPipe::kSlots, std::ref(slot));
  if (ran) *err = (hipError_t)first.load();
  return ran;
}

// All of [0, n): by `piece` on the workers, or, a few at a time while they
// are busy, by `plain` on this thread.
template <typename F, typename G>
hipError_t all_pieces(int device, size_t n, const F& piece, const G& plain) {
  size_t next[HostPipe::kSlots];
  for (size_t t = 0; t < HostPipe::kSlots; ++t) next[t] = t;
  hipError_t e = hipSuccess;
  for (bool left = true; left && e == hipSuccess;) {
    if (!pooled(device, n, next, piece, &e))
      for (size_t t = 0; t < HostPipe::kSlots && e == hipSuccess; ++t)
        if (next[t] < n) {
          e = plain(next[t], t);
          next[t] += HostPipe::kSlots;
        }
    left = false;
    for (size_t k : next) left = left || k < n;
  }
  return e;
}

}  // namespace

// The pipes of a device, asked to give their buffers back.  Its lock is not
// taken by a pipe in a transfer.
struct HostPipes {
  std::mutex mu;
  std::vector<HostPipe*> all;
};
static HostPipes& pipes_of(int device) {
  static std::mutex m;
  static std::map<int, HostPipes*> all;  // for the life of the process, as the memory managers
  std::lock_guard<std::mutex> g(m);
  auto it = all.find(device);
  if (it == all.end()) it = all.emplace(device, new HostPipes()).first;
  return *it->second;
}

// A transfer's use of the buffers.
struct HostPipe::Loan {
  HostPipe& p;
  const bool ok;
  Loan(HostPipe& pipe, int device, size_t bytes) : p(pipe), ok(pipe.begin(device, bytes)) {}
  ~Loan() {
    if (ok) p.end();
  }
};

bool HostPipe::begin(int device, size_t bytes) {
  if (device_ >= 0 && device_ != device) return false;
  {
    std::lock_guard<std::mutex> g(mu_);
    if (!buf_[0]) {
      if ((moved_ += bytes) < kWorth) return false;
      moved_ = 0;
    }
  }
  if (device_ < 0) {
    try {
      HostPipes& P = pipes_of(device);
      std::lock_guard<std::mutex> g(P.mu);
      P.all.push_back(this);
    } catch (const std::bad_alloc&) {
      return false;
    }
    device_ = device;
  }
  {
    std::lock_guard<std::mutex> g(mu_);
    busy_ = true;
  }
  if (buf_[0]) return true;
  // no room or no memory for the buffers: the runtime's path
  if (MemMan::ForDevice(device).ReserveSpareCPU(kSlots * kChunk, &HostPipe::give_back)) {
    bool ok = true;
    for (int i = 0; i < kSlots && ok; ++i)
      ok = hipHostMalloc(&buf_[i], kChunk, hipHostMallocDefault) == hipSuccess &&
           hipEventCreateWithFlags(&ev_[i], hipEventDisableTiming) == hipSuccess;
    if (ok) return true;
    (void)hipGetLastError();
    std::lock_guard<std::mutex> g(mu_);
    drop();
  }
  end();
  return false;
}

void HostPipe::end() {
  {
    std::lock_guard<std::mutex> g(mu_);
    busy_ = false;
  }
  idle_.notify_all();
}

void HostPipe::drop() {
  for (int i = 0; i < kSlots; ++i) {
    if (ev_[i]) {
      (void)hipEventSynchronize(ev_[i]);  // its last copy may still read the buffer
      (void)hipEventDestroy(ev_[i]);
    }
    if (buf_[i]) (void)hipHostFree(buf_[i]);
    ev_[i] = nullptr;
    buf_[i] = nullptr;
  }
  moved_ = 0;
  MemMan::ForDevice(device_).ReleaseSpareCPU(kSlots * kChunk);
}

void HostPipe::give(bool wait) {
  std::unique_lock<std::mutex> lk(mu_);
  if (busy_ && !wait) return;
  idle_.wait(lk, [&] { return !busy_; });
  if (buf_[0]) drop();
}

void HostPipe::give_back(int device, bool wait) {
  HostPipes& P = pipes_of(device);
  std::lock_guard<std::mutex> g(P.mu);
  for (HostPipe* p : P.all) p->give(wait);
}

void HostPipe::Release() {
  if (device_ >= 0) {
    HostPipes& P = pipes_of(device_);
    std::lock_guard<std::mutex> g(P.mu);
    P.all.erase(std::find(P.all.begin(), P.all.end(), this));
  }
  std::lock_guard<std::mutex> g(mu_);
  if (buf_[0]) drop();
  moved_ = 0;
  device_ = -1;
}

hipError_t HostPipe::Upload(int device, void* dst, const void* src, size_t bytes, hipStream_t stream) {
  if (bytes < kLeast || pinned(src)) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream);
  const Loan loan(*this, device, bytes);
  if (!loan.ok) return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, stream);
  hipError_t e = hipStreamSynchronize(stream);
  if (e != hipSuccess) return e;
  auto len = [&](size_t c) { return std::min(kChunk, bytes - c * kChunk); };
  auto piece = [&](size_t c, size_t t) {
    hipError_t q = hipEventSynchronize(ev_[t]);  // the buffer's last copy (an event never recorded is done)
    if (q != hipSuccess) return q;
    memcpy(buf_[t], (const char*)src + c * kChunk, len(c));
    q = hipMemcpyAsync((char*)dst + c * kChunk, buf_[t], len(c), hipMemcpyHostToDevice, stream);
    return q == hipSuccess ? hipEventRecord(ev_[t], stream) : q;
  };
  auto plain = [&](size_t c, size_t) {
    return hipMemcpyAsync((char*)dst + c * kChunk, (const char*)src + c * kChunk, len(c), hipMemcpyHostToDevice, stream);
  };
  e = all_pieces(device, (bytes + kChunk - 1) / kChunk, piece, plain);
  if (e != hipSuccess) (void)hipStreamSynchronize(stream);  // nothing reads the buffers any more
  return e;
}

hipError_t HostPipe::Download(int device, const CopyPiece* pieces, size_t n, hipStream_t stream) {
  size_t total = 0;
  bool direct = false;
  for (size_t i = 0; i < n; ++i) {
    total += pieces[i].bytes;
    direct = direct || pinned(pieces[i].dst);
  }
  auto by_runtime = [&] {
    for (size_t i = 0; i < n; ++i)
      if (hipError_t e = hipMemcpyAsync(pieces[i].dst, pieces[i].src, pieces[i].bytes, hipMemcpyDeviceToHost, stream))
        return e;
    return hipStreamSynchronize(stream);
  };
  if (total < kLeast || direct) return by_runtime();
  const Loan loan(*this, device, total);
  if (!loan.ok) return by_runtime();
  size_t m = 0;  // pieces of at most kChunk bytes, each of one image
  for (size_t i = 0; i < n; ++i) m += (pieces[i].bytes + kChunk - 1) / kChunk;
  auto cut = [&](size_t c) {
    size_t i = 0;
    for (size_t k; c >= (k = (pieces[i].bytes + kChunk - 1) / kChunk); c -= k) ++i;
    const size_t off = c * kChunk;
    return CopyPiece{(char*)pieces[i].dst + off, (const char*)pieces[i].src + off, std::min(kChunk, pieces[i].bytes - off)};
  };
  auto fetch = [&](size_t c, size_t t) {
    const CopyPiece p = cut(c);
    const hipError_t q = hipMemcpyAsync(buf_[t], p.src, p.bytes, hipMemcpyDeviceToHost, stream);
    return q == hipSuccess ? hipEventRecord(ev_[t], stream) : q;
  };
  auto drain = [&](size_t c, size_t t) {
    const CopyPiece p = cut(c);
    const hipError_t q = hipEventSynchronize(ev_[t]);
    if (q == hipSuccess) memcpy(p.dst, buf_[t], p.bytes);
    return q;
  };
  // each slot's first piece follows the stream's work at once; the workers
  // are taken when that work and the first piece are done
  const size_t ahead = std::min(m, (size_t)kSlots);
  hipError_t e = hipSuccess;
  for (size_t c = 0; c < ahead && e == hipSuccess; ++c) e = fetch(c, c);
  if (e == hipSuccess) e = hipEventSynchronize(ev_[0]);
  auto piece = [&](size_t c, size_t t) {
    const hipError_t q = c < ahead ? hipSuccess : fetch(c, t);
    return q == hipSuccess ? drain(c, t) : q;
  };
  bool queued = false;  // copies that nobody has waited for
  auto plain = [&](size_t c, size_t t) {
    if (c < ahead) return drain(c, t);
    const CopyPiece p = cut(c);
    queued = true;
    return hipMemcpyAsync(p.dst, p.src, p.bytes, hipMemcpyDeviceToHost, stream);
  };
  if (e == hipSuccess) e = all_pieces(device, m, piece, plain);
  if (e == hipSuccess && !queued) return e;  // every piece has been drained
  const hipError_t last = hipStreamSynchronize(stream);
  return e == hipSuccess ? last : e;
}

void parallel_memcpy(int device, void* dst, const void* src, size_t bytes) {
  constexpr size_t kPart = 1u << 20;
  const size_t n = (bytes + kPart - 1) / kPart;
  auto part = [&](size_t i) {
    const size_t off = i * kPart;
    memcpy((char*)dst + off, (const char*)src + off, std::min(kPart, bytes - off));
  };
  if (bytes < HostPipe::kLeast || !MemMan::ForDevice(device).TryParallelFor(n, HostPipe::kSlots, std::ref(part)))
    memcpy(dst, src, bytes);
}

}  // namespace tvk
