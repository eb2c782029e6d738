// Results on their way to the caller's memory.  A copy into pageable memory
// goes through the runtime's own staging, one piece after the other; here the
// pieces go through a few pinned buffers, so that the device fills one while
// the host empties another (BFS with its 16 KB result 112 -> 79 us, SSSP with
// 4 MB 1106 -> 1016, a batch with 224 MB in 52 arrays 65 -> 61 ms; what is left
// of the large ones is the first touch of the caller's pages).
#pragma once
#include <mutex>

#include "common.hpp"

namespace cg {

class HostStage {
 public:
  HostStage() = default;
  HostStage(const HostStage&) = delete;
  HostStage& operator=(const HostStage&) = delete;
  ~HostStage() {
    for (auto& s : slot_)
      if (s.ev) (void)hipEventDestroy(s.ev);
  }

  // The first buffer for results of n bytes, so that the first one does not
  // wait for a pinned allocation (50-90 us).
  int prepare(size_t n) { return fill(slot_[0], n < kPiece ? n : kPiece); }

  // Results of up to this size go through pinned memory that the owner has
  // anyway and lends: no allocation (BFS of 4096 vertices 178 -> 140 us to create).
  static constexpr size_t kSmall = 1u << 18;
  int lend(uint8_t* p, size_t n) {
    slot_[0].p = p;
    slot_[0].cap = n;
    return fill(slot_[0], n);
  }

  // Queues a copy of n bytes behind the stream's work.  The bytes are in dst
  // once finish() has returned.
  int put(void* dst, const void* src, size_t n, hipStream_t s) {
    if (!n) return CG_OK;
    // memory the device reaches (pinned, managed): no detour
    hipPointerAttribute_t a{};
    if (hipPointerGetAttributes(&a, dst) != hipSuccess) (void)hipGetLastError();
    else if (a.type != hipMemoryTypeUnregistered) {
      CG_HIP(hipMemcpyAsync(dst, src, n, hipMemcpyDeviceToHost, s));
      direct_ = true;
      return CG_OK;
    }
    for (size_t o = 0; o < n; o += kPiece) {
      const size_t m = n - o < kPiece ? n - o : kPiece;
      Slot& t = slot_[next_];
      CG_TRY(empty(t));
      CG_TRY(fill(t, m));
      CG_HIP(hipMemcpyAsync(t.p, static_cast<const uint8_t*>(src) + o, m, hipMemcpyDeviceToHost, s));
      CG_HIP(hipEventRecord(t.ev, s));
      t.dst = static_cast<uint8_t*>(dst) + o;
      t.n = m;
      next_ = (next_ + 1) % kSlots;
    }
    return CG_OK;
  }

  int finish(hipStream_t s) {
    for (int i = 0; i < kSlots; ++i) CG_TRY(empty(slot_[(next_ + i) % kSlots]));
    if (direct_) CG_HIP(hipStreamSynchronize(s));
    direct_ = false;
    next_ = 0;  // one piece at a time takes one buffer
    return CG_OK;
  }

  // After an error: waits for the copies under way and forgets them.
  void drop(hipStream_t s) {
    (void)hipStreamSynchronize(s);
    for (auto& t : slot_) t.n = 0;
    direct_ = false;
    next_ = 0;
  }

  std::mutex mu;  // a stage serves one call at a time

 private:
  // (SSSP with 4 MB: pieces of 256 KB / 512 KB / 1 / 2 / 4 MB 1133 / 1033 / 1000 / 1020 / 1052 us)
  static constexpr size_t kPiece = 1u << 20;
  static constexpr int kSlots = 3;
  struct Slot {
    PinnedBuf<uint8_t> buf;
    uint8_t* p = nullptr;  // buf's or lent
    size_t cap = 0;
    hipEvent_t ev = nullptr;
    void* dst = nullptr;
    size_t n = 0;
  };
  static int fill(Slot& t, size_t n) {
    if (t.cap < n) {
      t.cap = 0;
      CG_TRY(t.buf.ensure(n));
      t.p = t.buf.p;
      t.cap = n;
    }
    if (!t.ev) CG_HIP(hipEventCreateWithFlags(&t.ev, hipEventDisableTiming));
    return CG_OK;
  }
  int empty(Slot& t) {
    if (!t.n) return CG_OK;
    CG_HIP(hipEventSynchronize(t.ev));
    std::memcpy(t.dst, t.p, t.n);
    t.n = 0;
    return CG_OK;
  }
  Slot slot_[kSlots];
  int next_ = 0;
  bool direct_ = false;
};

}  // namespace cg
