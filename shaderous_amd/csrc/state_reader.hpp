// Reading a state back to ordinary host memory. hipMemcpyAsync into pageable memory moves about
// 9.5 GB/s here: one thread touches the destination's pages and copies from the runtime's staging.
// So a large state goes in chunks through pinned slots of the sim's own, one host thread per slot:
// while a chunk crosses the bus, other threads copy theirs out (and take its page faults). 268 MiB
// take 30 ms plain and 6.4 ms with 8 slots of 4 MiB (43 GB/s; slots of 2 MiB give 39, of 1 MiB 31,
// four slots of 4 MiB 37).
// By the state's size, plain -> here, into memory used before and into fresh memory:
//   32 MiB 1.95 -> 0.95 and 3.8 -> 1.2 ms, 8 MiB 0.96 -> 0.36 and 1.4 -> 0.60 ms: threads;
//   6 MiB 0.41 -> 0.53 and 1.5 -> 0.58 ms, 2 MiB 0.13 -> 0.14 and 0.49 -> 0.31 ms: starting the
//   threads costs what they save where the pages are there already, so plain copies up to 8 MiB;
//   128 KiB 0.074 -> 0.026 and 0.098 -> 0.045 ms, 512 KiB 0.043 and 0.14 -> 0.12 ms: up to 512 KiB
//   both arrays through one slot, with no thread.
// A pinned or device destination takes the plain copy, which is then direct.
#pragma once
#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <mutex>
#include <thread>

namespace shx {

class StateReader {
 public:
  static constexpr int SLOTS = 8;
  static constexpr size_t LEAST = (size_t)512 << 10;   // states read through one slot
  static constexpr size_t MOST = (size_t)4 << 20;      // bytes per slot
  static constexpr size_t LARGE = (size_t)8 << 20;     // states read by several threads

  ~StateReader() { drop(); }

  // Slots for states of `least` to `most` bytes: 8 (at most half the host's threads) of a 16th of the
  // largest, 1 to 4 MiB, where there are large ones, else one for the small ones if there are any.
  // Pinned memory costs: 0.05 ms for the least of it, a quarter of the time in which a small sim is made
  // (one read through it saves as much), and the first touch of its pages, on the first read. States of
  // 16 and 32 MiB take 2.2 and 3.0 ms on their first read with slots twice as large, 1.0 and 1.8 with
  // these; 0.53 and 0.89 against 0.59 and 0.92 on later ones. Without memory for them reads are plain
  // copies.
  void fit(size_t least, size_t most) {
    if (least > LEAST && most < LARGE) return;
    const unsigned int hw = std::thread::hardware_concurrency();
    const int n = most < LARGE ? 1 : std::max(1, std::min(SLOTS, (int)(hw / 2)));
    const size_t per = most < LARGE ? std::min(LEAST, (most + 4095) & ~(size_t)4095)
                                    : std::min(MOST, std::max((size_t)1 << 20, most / 16));
    if (n <= count_ && per <= (n == 1 ? room() : 2 * chunk_)) return;
    drop();
    if (hipHostMalloc((void**)&pinned_, n * per, hipHostMallocDefault) != hipSuccess) {
      (void)hipGetLastError();
      pinned_ = nullptr;
      return;
    }
    chunk_ = per;
    for (; count_ < n; count_++)
      if (hipEventCreateWithFlags(&done_[count_], hipEventDisableTiming) != hipSuccess) {
        (void)hipGetLastError();
        break;
      }
  }

  // Two arrays of `bytes` each, in stream order; returns when both are there. Reads of one sim take
  // their turns.
  hipError_t read(hipStream_t stream, int device, void* d0, const void* s0, void* d1, const void* s1, size_t bytes) {
    const bool small = 2 * bytes <= std::min(LEAST, room());
    if (count_ == 0 || (!small && (count_ == 1 || 2 * bytes < LARGE)) || !pageable(d0) || !pageable(d1)) {
      hipError_t e = hipMemcpyAsync(d0, s0, bytes, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipMemcpyAsync(d1, s1, bytes, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
      return e;
    }
    std::lock_guard<std::mutex> lock(mutex_);
    if (small) {
      hipError_t e = hipMemcpyAsync(pinned_, s0, bytes, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipMemcpyAsync(pinned_ + bytes, s1, bytes, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
      if (e != hipSuccess) return e;
      memcpy(d0, pinned_, bytes);
      memcpy(d1, pinned_ + bytes, bytes);
      return hipSuccess;
    }
    const size_t each = (bytes + chunk_ - 1) / chunk_;   // chunks per array
    std::atomic<size_t> next{0};
    std::atomic<int> bad{(int)hipSuccess};
    auto work = [&](int w) {
      hipError_t e = w == 0 ? hipSuccess : hipSetDevice(device);
      for (size_t c; e == hipSuccess && bad == (int)hipSuccess && (c = next++) < 2 * each;) {
        const size_t off = (c % each) * chunk_, n = std::min(chunk_, bytes - off);
        char* slot = pinned_ + w * chunk_;
        e = hipMemcpyAsync(slot, (const char*)(c < each ? s0 : s1) + off, n, hipMemcpyDeviceToHost, stream);
        if (e == hipSuccess) e = hipEventRecord(done_[w], stream);
        if (e == hipSuccess) e = hipEventSynchronize(done_[w]);
        if (e == hipSuccess) memcpy((char*)(c < each ? d0 : d1) + off, slot, n);
      }
      if (e != hipSuccess) bad = (int)e;
    };
    std::thread others[SLOTS];
    const int n = (int)std::min<size_t>(count_, 2 * each);
    for (int w = 1; w < n; w++) {
      try {
        others[w] = std::thread(work, w);
      } catch (...) {
        break;   // no thread, or no memory for one: fewer do it too
      }
    }
    work(0);
    for (int w = 1; w < n; w++)
      if (others[w].joinable()) others[w].join();
    if (bad != (int)hipSuccess) (void)hipStreamSynchronize(stream);   // no copy still under way
    return (hipError_t)bad.load();
  }

 private:
  static bool pageable(const void* p) {
    if (!p) return false;
    hipPointerAttribute_t a;
    if (hipPointerGetAttributes(&a, p) != hipSuccess) {
      (void)hipGetLastError();
      return true;
    }
    return a.type == hipMemoryTypeUnregistered;
  }
  size_t room() const { return count_ * chunk_; }
  void drop() {
    for (; count_ > 0; count_--) (void)hipEventDestroy(done_[count_ - 1]);
    if (pinned_) (void)hipHostFree(pinned_);
    pinned_ = nullptr;
    chunk_ = 0;
  }

  std::mutex mutex_;
  char* pinned_ = nullptr;
  size_t chunk_ = 0;
  int count_ = 0;
  hipEvent_t done_[SLOTS] = {};
};

}  // namespace shx
