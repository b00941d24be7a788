// The copies between host and device memory (ac_stage.hpp) on the CPU: the HIP calls they make are stood in for here by a
// queue of copies that are carried out, in order, only when something waits for them.  Prints "0 failed checks".
#include <hip/hip_runtime_api.h>

#include <cstdio>
#include <deque>
#include <map>
#include <mutex>
#include <set>
#include <vector>

#include "../application_classification_amd/csrc/ac_stage.hpp"

namespace {
struct Op {
  void* dst;
  const void* src;
  size_t bytes;
  hipEvent_t ev;  // or a recorded event
};
std::mutex mu;
std::deque<Op> queue;
std::set<const void*> known;  // memory that HIP knows
size_t pinned = 0;
int copies = 0, selects = 0, wrong_device = 0, failed = 0;
bool no_pinned = false, fail_copies = false;
thread_local int device = 0;
const hipStream_t kStream = reinterpret_cast<hipStream_t>(8);

void drain(hipEvent_t until) {
  std::lock_guard<std::mutex> l(mu);
  while (!queue.empty()) {
    const Op o = queue.front();
    queue.pop_front();
    if (o.bytes) std::memcpy(o.dst, o.src, o.bytes);
    if (until && o.ev == until) break;
  }
}
#define CHECK(x)                                             \
  do {                                                       \
    if (!(x)) ++failed, std::printf("line %d: %s\n", __LINE__, #x); \
  } while (0)
}  // namespace

extern "C" {
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  *e = reinterpret_cast<hipEvent_t>(new char);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
  delete reinterpret_cast<char*>(e);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  if (no_pinned) return hipErrorOutOfMemory;
  *p = new char[n];
  pinned += n;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  delete[] static_cast<char*>(p);
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipSetDevice(int d) {
  device = d;
  std::lock_guard<std::mutex> l(mu);
  ++selects;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  if (!known.count(p)) return hipErrorInvalidValue;
  a->type = hipMemoryTypeHost;
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, hipMemcpyKind, hipStream_t) {
  std::lock_guard<std::mutex> l(mu);
  if (fail_copies) return hipErrorUnknown;
  ++copies;
  wrong_device += device != 1;
  queue.push_back(Op{dst, src, bytes, nullptr});
  return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) {
  std::lock_guard<std::mutex> l(mu);
  queue.push_back(Op{nullptr, nullptr, 0, e});
  return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e) {
  {
    std::lock_guard<std::mutex> l(mu);
    bool there = false;
    for (const Op& o : queue) there = there || o.ev == e;
    if (!there) return hipSuccess;
  }
  drain(e);
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) {
  drain(nullptr);
  return hipSuccess;
}
}

int main() {
  using ac::HostStage;
  device = 1;
  const size_t sizes[] = {1, 4096, HostStage::kSmall, HostStage::kSmall + 1, HostStage::kDirect - 1, HostStage::kDirect,
                          (5 << 20) + 3, (16 << 20) - 1, 16 << 20, (19 << 20) + 7};
  auto fill = [](std::vector<char>& v, int seed) {
    for (size_t i = 0; i < v.size(); ++i) v[i] = (char)(i * 31 + i / 4099 + seed);
  };
  for (const bool none : {false, true})
    for (const size_t n : sizes) {
      no_pinned = none;
      HostStage s;
      std::vector<char> a(n), b(n, 0), c(n, 0);
      fill(a, 1);
      pinned = 0, copies = selects = wrong_device = 0;
      // Inputs: two in a row, the source overwritten after each, before anything has waited.
      const std::vector<char> first = a;
      CHECK(s.to_device(b.data(), a.data(), n, kStream) == hipSuccess);
      fill(a, 2);
      const std::vector<char> second = a;
      CHECK(s.to_device(c.data(), a.data(), n, kStream) == hipSuccess);
      fill(a, 3);
      drain(nullptr);
      CHECK(b == first);
      CHECK(c == second);
      // Small inputs pin a small buffer, ones in between none, large ones the slots.
      const size_t all = HostStage::kSlots * HostStage::kSlot;
      CHECK(pinned == (none ? 0 : n <= HostStage::kSmall ? HostStage::kSmall : n < HostStage::kDirect ? 0 : all));
      // Results, into pageable memory: complete on return, every item of the copy on the context's device.
      std::vector<char> d(n, 0);
      copies = selects = 0;
      CHECK(s.to_host(d.data(), a.data(), n, kStream, 1) == hipSuccess);
      CHECK(d == a);
      CHECK(wrong_device == 0);
      const bool staged = !none && n >= HostStage::kDirect;
      CHECK(copies == 1 ? !staged : staged);
      CHECK(!staged || selects == (n < (16u << 20) ? 1 : HostStage::kThreads));
      // Into and out of memory that HIP knows: one copy, complete on return.
      for (auto& x : d) x = 0;
      known = {d.data(), a.data()};
      copies = 0;
      CHECK(s.to_host(d.data(), a.data(), n, kStream, 1) == hipSuccess && copies == 1 && d == a);
      for (auto& x : b) x = 0;
      CHECK(s.to_device(b.data(), a.data(), n, kStream) == hipSuccess && copies == 2 && b == a);
      known.clear();
      // An error of a copy is the call's, and the next call works.
      fail_copies = true;
      CHECK(s.to_host(d.data(), a.data(), n, kStream, 1) != hipSuccess);
      CHECK(s.to_device(b.data(), a.data(), n, kStream) != hipSuccess);
      fail_copies = false;
      fill(a, 4);
      CHECK(s.to_host(d.data(), a.data(), n, kStream, 1) == hipSuccess && d == a);
    }
  std::printf("%d failed checks\n", failed);
  return failed != 0;
}
