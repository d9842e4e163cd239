// CPU check of csrc/fetch.hpp against a HIP runtime that this file plays: copies
// into pinned memory run no earlier than the wait that promises them, their
// targets hold rubbish until then, and pinning can be made to fail.
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "fetch.hpp"

namespace {
struct Copy {
  void* dst;
  const void* src;
  size_t bytes;
};
std::mutex gLock;
std::map<char*, size_t> gPinned;  // live pinned blocks
int gEvents = 0;                  // live events
constexpr int kAny = 1 << 20;
int gLanes = 0, gLaneLimit = kAny, gMostLanes = 0;  // pinned lanes of 2 MiB: now, allowed, at most
int gCopies = 0, gCopyLimit = kAny;
std::vector<Copy> gQueue;
size_t gDone = 0;
thread_local int tDevice = 0;
thread_local hipError_t tLast = hipSuccess;

void runTo(size_t k) {
  for (; gDone < k; gDone++)
    if (const Copy& c = gQueue[gDone]; c.bytes) std::memcpy(c.dst, c.src, c.bytes);
}
bool pinned(void* p) {
  auto it = gPinned.upper_bound(static_cast<char*>(p));
  if (it == gPinned.begin()) return false;
  --it;
  return static_cast<char*>(p) < it->first + it->second;
}
struct Event {
  size_t at;
  int device;
};
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) {
  *d = tDevice;
  return hipSuccess;
}
hipError_t hipSetDevice(int d) {
  tDevice = d;
  return hipSuccess;
}
hipError_t hipGetLastError(void) {
  const hipError_t e = tLast;
  tLast = hipSuccess;
  return e;
}
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned int) {
  std::lock_guard<std::mutex> g(gLock);
  const int lanes = int(bytes >> 21);
  if (gLanes + lanes > gLaneLimit) return tLast = hipErrorOutOfMemory;
  gLanes += lanes;
  gMostLanes = std::max(gMostLanes, gLanes);
  *p = std::malloc(bytes);
  gPinned[static_cast<char*>(*p)] = bytes;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  std::lock_guard<std::mutex> g(gLock);
  gLanes -= int(gPinned[static_cast<char*>(p)] >> 21);
  gPinned.erase(static_cast<char*>(p));
  std::free(p);
  return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  std::lock_guard<std::mutex> g(gLock);
  gEvents++;
  *e = reinterpret_cast<hipEvent_t>(new Event{0, tDevice});
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> g(gLock);
  gEvents--;
  delete reinterpret_cast<Event*>(e);
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> g(gLock);
  Event* v = reinterpret_cast<Event*>(e);
  if (v->device != tDevice) return hipErrorInvalidHandle;
  v->at = gQueue.size();
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  std::lock_guard<std::mutex> g(gLock);
  runTo(reinterpret_cast<Event*>(e)->at);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  std::lock_guard<std::mutex> g(gLock);
  runTo(gQueue.size());
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t) {
  std::lock_guard<std::mutex> g(gLock);
  if (gCopies >= gCopyLimit) return hipErrorUnknown;
  gCopies++;
  if (pinned(dst)) {
    gQueue.push_back({dst, src, bytes});
    std::memset(dst, 0xFF, bytes);
  } else if (bytes) {
    std::memcpy(dst, src, bytes);  // pageable memory: the call returns when the copy is done
  }
  return hipSuccess;
}
}

namespace {
int gBad = 0;
void check(bool ok, const char* what, size_t n) {
  if (ok) return;
  gBad++;
  std::printf("FAILED: %s (n %zu)\n", what, n);
}

template <class T>
hipError_t fetched(kofm::FetchStage& s, size_t n, bool& same) {
  std::vector<T> src(n);
  uint32_t v = uint32_t(n) + 12345u;
  for (auto& x : src) {
    v = v * 1664525u + 1013904223u;
    x = T(double(int32_t(v)) / 65536.);
  }
  std::vector<double> out(n + 2, -7.);
  const hipError_t e = s.fetch(hipStream_t(nullptr), src.data(), n, out.data() + 1);
  same = out.front() == -7. && out.back() == -7.;
  for (size_t i = 0; i < n && same; i++) same = out[i + 1] == double(src[i]);
  gQueue.clear();
  gDone = 0;
  return e;
}
template <class T>
void expect(kofm::FetchStage& s, size_t n, const char* what) {
  bool same = false;
  check(fetched<T>(s, n, same) == hipSuccess, what, n);
  check(same, what, n);
}

constexpr size_t kMiB = size_t(1) << 20;
const size_t kLarge = 33 * kMiB + 4 * 1001;  // bytes of a field that takes every lane it can get

void open(kofm::FetchStage& s, size_t largest = kLarge) {
  check(s.open(largest) == hipSuccess, "open", largest);
}

template <class T>
void sizes() {
  const size_t piece = kMiB / sizeof(T);
  for (size_t n : {size_t(0), size_t(1), size_t(77), piece - 1, piece, piece + 1, 2 * piece, 2 * piece + 1,
                   3 * piece - 1, 4 * piece - 1, 4 * piece, 4 * piece + 5, 8 * piece - 1, 8 * piece,
                   8 * piece + 3, 17 * piece + 11, 33 * piece + 7}) {
    kofm::FetchStage s;
    open(s);
    expect<T>(s, n, "a field");
    expect<T>(s, n, "the same field again");
  }
}
void allGivenBack() { check(gPinned.empty() && gEvents == 0, "everything given back", gPinned.size()); }
}  // namespace

int main() {
  {  // contexts share what the first has pinned for its largest field
    kofm::FetchStage s[48], small;
    open(small, 1000);
    check(gLanes == 1, "one lane for a small lattice", size_t(gLanes));
    for (auto& x : s) open(x);
    check(gLanes == 4, "four lanes for large ones, however many", size_t(gLanes));
    for (auto& x : s) expect<float>(x, kLarge / 4, "a large FP32 field");
    expect<double>(small, 1000, "a small field");
    expect<double>(s[0], kLarge / 8, "a large field");
    check(gLanes == 4, "nothing pinned for contexts read in turn", size_t(gLanes));
  }
  allGivenBack();

  sizes<float>();
  sizes<double>();
  allGivenBack();

  for (int lanes : {0, 1, 2, 3}) {  // pinning fails: at once, or from some lane on
    kofm::FetchStage s;
    gLaneLimit = lanes;
    open(s);
    expect<float>(s, kLarge / 4 + 1, "FP32 with lanes missing");
    expect<double>(s, kLarge / 8 + 1, "FP64 with lanes missing");
    expect<float>(s, 1, "one value with lanes missing");
    check(tLast == hipSuccess, "the refusal is not left for the next call", size_t(lanes));
    check(gLanes <= lanes, "lanes missing", size_t(gLanes));
    gLaneLimit = kAny;
    expect<float>(s, kLarge / 4 + 1, "lanes pinned later");
    check(gLanes == 4, "lanes pinned later", size_t(gLanes));
  }
  allGivenBack();

  {  // two devices: each has lanes (and events) of its own
    kofm::FetchStage a, b;
    tDevice = 3;
    open(a);
    tDevice = 1;
    open(b);
    expect<float>(b, kLarge / 4, "the second device");
    tDevice = 3;
    expect<float>(a, kLarge / 4, "the first device");
    check(gEvents == 16, "lanes of two devices", size_t(gEvents));
    tDevice = 0;
  }
  allGivenBack();

  {  // twenty threads, each reading its own context: no lane is used twice at a time
    gMostLanes = 0;
    std::vector<std::thread> team;
    std::atomic<int> wrong{0};
    std::vector<float> src(kLarge / 4);
    for (size_t i = 0; i < src.size(); i++) src[i] = float(i % 1000003);
    for (int t = 0; t < 20; t++)
      team.emplace_back([&, t] {
        kofm::FetchStage s;
        if (s.open(kLarge) != hipSuccess) wrong++;
        const size_t off = size_t(t) * 1009, n = src.size() - off;
        std::vector<double> out(n);
        for (int r = 0; r < 3; r++) {
          std::fill(out.begin(), out.end(), -1.);
          if (s.fetch(hipStream_t(nullptr), src.data() + off, n, out.data()) != hipSuccess) wrong++;
          for (size_t i = 0; i < n; i++)
            if (out[i] != double(src[off + i])) {
              wrong++;
              break;
            }
        }
      });
    for (auto& t : team) t.join();
    check(wrong == 0, "contexts read at the same time", size_t(wrong));
    check(gMostLanes <= 16, "a bounded number of lanes", size_t(gMostLanes));
    gQueue.clear();
    gDone = 0;
  }
  allGivenBack();

  for (int k = 0; k < 12; k++) {  // the k-th copy fails: an error, and the stage still works
    kofm::FetchStage s;
    open(s);
    gCopies = 0;
    gCopyLimit = k;
    bool same = false;
    check(fetched<double>(s, kLarge / 8, same) != hipSuccess, "a failing copy is reported", size_t(k));
    gCopyLimit = kAny;
    expect<double>(s, kLarge / 8, "after a failed copy");
  }
  allGivenBack();
  std::printf(gBad ? "%d checks failed\n" : "ok\n", gBad);
  return gBad ? 1 : 0;
}
