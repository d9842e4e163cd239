// fetch.hpp -- fields on their way from the device to the caller's doubles.
#pragma once

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace kofm {

// Pinned host memory of one device, in lanes of two pieces of 1 MiB, shared by
// the contexts on it.  The first context pins what its largest field takes, 2
// or 8 MiB; later ones find it there (each for itself, 48 channels held
// 384 MiB), and only contexts read at the same time, from threads of their own,
// pin more, up to kMost lanes.  All are given back with the device's last
// context.  Pinned by the contexts' creation, not by their first field: a
// context alone on its device pays 0.05 ms there, and paid 0.1 to 1.2 ms with
// the field (2048 x 256: 0.28 ms became 1.25).  Shared, the first reading of
// six channels' 30 fields went from 15.9 to 12.2 ms, 16 steps included.
class PinnedLanes {
 public:
  static constexpr size_t kPiece = size_t(1) << 20;
  static constexpr int kMost = 16;
  struct Lane {
    char* mem = nullptr;
    hipEvent_t done[2] = {};
    char* block = nullptr;  // to be freed (the first lane of an allocation)
  };

  // The lanes of a device, alive while somebody holds them.
  static std::shared_ptr<PinnedLanes> of(int device) {
    static std::mutex& lock = *new std::mutex;  // (not destroyed before a late context)
    static auto& all = *new std::map<int, std::weak_ptr<PinnedLanes>>;
    std::lock_guard<std::mutex> guard(lock);
    std::shared_ptr<PinnedLanes> p = all[device].lock();
    if (!p) all[device] = p = std::make_shared<PinnedLanes>(device);
    return p;
  }

  explicit PinnedLanes(int device) : device_(device) { free_.reserve(kMost); }
  PinnedLanes(const PinnedLanes&) = delete;
  PinnedLanes& operator=(const PinnedLanes&) = delete;
  ~PinnedLanes() {
    for (Lane& l : lanes_) drop(l);
  }

  // Sees to it that n lanes exist, where they can be pinned.
  void reserve(int n) {
    std::lock_guard<std::mutex> guard(lock_);
    for (int m = made_, end = m + make(n - m); m < end; m++) free_.push_back(&lanes_[m]);
  }

  // Up to `want` lanes that nobody uses; the number taken (0 when all are in
  // use or none can be pinned).
  int take(int want, Lane** out) {
    std::lock_guard<std::mutex> guard(lock_);
    int n = 0;
    for (; n < want && !free_.empty(); n++) {
      out[n] = free_.back();
      free_.pop_back();
    }
    for (int m = made_, end = m + make(want - n); m < end; m++) out[n++] = &lanes_[m];
    return n;
  }
  void give(int n, Lane** lanes) {
    std::lock_guard<std::mutex> guard(lock_);
    while (n-- > 0) free_.push_back(lanes[n]);
  }

 private:
  const int device_;
  std::mutex lock_;
  Lane lanes_[kMost];
  int made_ = 0;
  std::vector<Lane*> free_;

  // The lanes' device as the calling thread's current one, for a while.
  struct Device {
    int mine, before;
    bool ok;
    explicit Device(int d) : mine(d), before(d) {
      ok = hipGetDevice(&before) == hipSuccess && (before == mine || hipSetDevice(mine) == hipSuccess);
    }
    ~Device() {
      if (before != mine) (void)hipSetDevice(before);
    }
  };

  // Makes up to n more lanes, in one allocation where that succeeds (four cost
  // as much as all else in a small context); the number made.
  int make(int n) {
    n = std::min(n, kMost - made_);
    if (n <= 0) return 0;
    const Device here(device_);
    if (!here.ok) return 0;
    char* block = nullptr;
    for (; n > 0; n /= 2) {
      if (hipHostMalloc(reinterpret_cast<void**>(&block), 2 * kPiece * size_t(n), hipHostMallocDefault) ==
          hipSuccess)
        break;
      (void)hipGetLastError();  // handled here: the field goes another way
    }
    for (int i = 0; i < n; i++) {
      Lane& l = lanes_[made_];
      l.mem = block + 2 * kPiece * size_t(i);
      if (i == 0) l.block = block;
      for (hipEvent_t& ev : l.done)
        if (hipEventCreateWithFlags(&ev, hipEventDisableTiming) != hipSuccess) {
          (void)hipGetLastError();
          drop(l);
          return i;
        }
      made_++;
    }
    return n;
  }
  static void drop(Lane& l) {
    for (hipEvent_t ev : l.done)
      if (ev) (void)hipEventDestroy(ev);
    if (l.block) (void)hipHostFree(l.block);
    l = Lane{};
  }
};

// The way of a context's fields: through a lane piece by piece, so that one
// piece is converted or copied out while the next one arrives.  Fields of
// 8 MiB (on the device) and more go through four lanes, a host thread each: a
// single thread is bound by the page faults of the caller's fresh arrays.  The
// line lies where that first pays.  One lane against four, us a field, into an
// array whose pages are there and, in brackets, three fields into new pages:
// FP32 4 MiB 176 and 236, 8 MiB 318 and 400 (2480 and 2080), 12 MiB 466 and 508
// (5280 and 2990); FP64 6 MiB 268 and 308 (2130 and 1420), 8 MiB 328 and 341,
// 16 MiB 646 and 602.  A field of 8192 x 1024 took 12 ms through an unpinned copy
// and a conversion, 2.2 ms this way; 2001 x 203 0.20 and 0.14 ms.  Without a lane
// a field is copied unpinned.
class FetchStage {
 public:
  // The stage of a context on the current device whose largest field has so
  // many bytes there.
  hipError_t open(size_t largest) {
    const hipError_t e = hipGetDevice(&device_);
    if (e != hipSuccess) return e;
    pinned_ = PinnedLanes::of(device_);
    pinned_->reserve(lanesFor(largest));
    return e;
  }

  // n values of type T at the device address src to doubles at host, after
  // the work enqueued on stream.
  template <class T>
  hipError_t fetch(hipStream_t stream, const T* src, size_t n, double* host) {
    Lane* l[kLanes];
    const int lanes = pinned_->take(lanesFor(n * sizeof(T)), l);
    if (lanes == 0) return unpinned(stream, src, n, host);
    std::atomic<int> bad{int(hipSuccess)};
    auto part = [&](int t) {
      const size_t a = n * size_t(t) / size_t(lanes), b = n * size_t(t + 1) / size_t(lanes);
      const hipError_t e = through(*l[t], stream, src, a, b, host);
      if (e != hipSuccess) bad = int(e);
    };
    std::thread team[kLanes];
    int started = 1;
    try {
      for (; started < lanes; started++)
        team[started] = std::thread([&, t = started] {
          if (hipSetDevice(device_) == hipSuccess)
            part(t);
          else
            bad = int(hipErrorInvalidDevice);
        });
    } catch (const std::system_error&) {  // no more threads: the rest runs here
    }
    part(0);
    for (int t = started; t < lanes; t++) part(t);
    for (int t = 1; t < started; t++) team[t].join();
    pinned_->give(lanes, l);
    return hipError_t(bad.load());
  }

 private:
  using Lane = PinnedLanes::Lane;
  static constexpr size_t kLaneFrom = size_t(8) << 20;
  static constexpr int kLanes = 4;
  std::shared_ptr<PinnedLanes> pinned_;
  int device_ = 0;

  static int lanesFor(size_t bytes) { return bytes >= kLaneFrom ? kLanes : 1; }

  // Values a .. b - 1 through one lane.
  template <class T>
  static hipError_t through(const Lane& l, hipStream_t stream, const T* src, size_t a, size_t b,
                            double* host) {
    constexpr size_t per = PinnedLanes::kPiece / sizeof(T);
    T* buf[2] = {reinterpret_cast<T*>(l.mem), reinterpret_cast<T*>(l.mem + PinnedLanes::kPiece)};
    auto start = [&](size_t i, int k) {
      hipError_t e = hipMemcpyAsync(buf[k], src + i, std::min(per, b - i) * sizeof(T),
                                    hipMemcpyDeviceToHost, stream);
      return e == hipSuccess ? hipEventRecord(l.done[k], stream) : e;
    };
    if (b - a <= per) {
      hipError_t e = hipMemcpyAsync(buf[0], src + a, (b - a) * sizeof(T), hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipStreamSynchronize(stream);
      if (e == hipSuccess) std::copy(buf[0], buf[0] + (b - a), host + a);
      return e;
    }
    hipError_t e = start(a, 0);
    int k = 0;
    for (size_t i = a; i < b && e == hipSuccess; i += per, k ^= 1) {
      if (i + per < b) e = start(i + per, k ^ 1);
      if (e == hipSuccess) e = hipEventSynchronize(l.done[k]);
      if (e == hipSuccess) std::copy(buf[k], buf[k] + std::min(per, b - i), host + i);
    }
    // nothing may still be arriving when the lane is used again
    if (e != hipSuccess) (void)hipStreamSynchronize(stream);
    return e;
  }

  // The values into the end of the caller's array, then widened from there:
  // host[i] ends before value i + 1 begins.
  template <class T>
  static hipError_t unpinned(hipStream_t stream, const T* src, size_t n, double* host) {
    char* tail = reinterpret_cast<char*>(host) + n * (sizeof(double) - sizeof(T));
    hipError_t e = hipMemcpyAsync(tail, src, n * sizeof(T), hipMemcpyDeviceToHost, stream);
    if (e == hipSuccess) e = hipStreamSynchronize(stream);
    if (e != hipSuccess || sizeof(T) == sizeof(double)) return e;
    for (size_t i = 0; i < n; i++) {
      T v;
      std::memcpy(&v, tail + i * sizeof(T), sizeof(T));
      host[i] = double(v);
    }
    return e;
  }
};

}  // namespace kofm
