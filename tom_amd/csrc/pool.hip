// Device workspaces kept between calls.
//
// A call such as tom_os3_corr on 256x256x128 takes 24 workspaces, 0.9 GB in
// all, and gave them back to the driver at its end: 3 to 24 ms of hipMalloc
// and hipFree (it differs from machine to machine) around 0.95 ms of kernels.
// Here a freed workspace waits for the next request of its size. It carries
// an event recorded on the stream that used it last, which the next request
// waits for whatever stream it names (equal handles may be different streams),
// so calls on several streams and threads may share the pool. At most kKeep
// bytes wait per device, oldest out first; all of it goes when an allocation
// of this library fails, when tomhip_release_workspaces asks for it or when the
// device's last context is destroyed.
#include <map>
#include <mutex>
#include <vector>

#include "common.h"
#include "pool.h"

namespace tomhip {

namespace {

constexpr size_t kKeep = 4ull << 30;

struct Block {
  void* p = nullptr;
  size_t size = 0;
  hipEvent_t ev = nullptr;
  bool idle = true;  // nothing queued uses it
};

struct Device {
  std::vector<Block> kept;  // oldest first
  size_t bytes = 0;
  int contexts = 0;
};

struct State {
  std::mutex mu;
  std::map<int, Device> dev;
  std::map<const void*, std::pair<int, Block>> used;
};
State& state() {
  static State* s = new State;  // outlives every static destructor
  return *s;
}

void drop(Block& b) {
  (void)hipFree(b.p);
  if (b.ev) (void)hipEventDestroy(b.ev);
}
void drop_all(Device& d) {
  for (Block& b : d.kept) drop(b);
  d.kept.clear();
  d.bytes = 0;
}

void* malloc_or_drop(Device& d, size_t bytes) {
  void* p = nullptr;
  hipError_t e = hipMalloc(&p, bytes);
  if (e != hipSuccess && !d.kept.empty()) {
    (void)hipGetLastError();
    drop_all(d);
    e = hipMalloc(&p, bytes);
  }
  TOMHIP_CHECK(e);
  return p;
}

size_t rounded(size_t n) {
  const size_t step = n < (1u << 20) ? 4096 : (1u << 20);
  return (n + step - 1) / step * step;
}

void keep(int device, Block b) {
  State& S = state();
  Device& d = S.dev[device];
  if (b.size > kKeep || d.contexts == 0) {
    drop(b);
    return;
  }
  while (!d.kept.empty() && d.bytes + b.size > kKeep) {
    d.bytes -= d.kept.front().size;
    drop(d.kept.front());
    d.kept.erase(d.kept.begin());
  }
  d.bytes += b.size;
  d.kept.push_back(b);
}

// what may still use a block that is given back
enum Use { U_NONE, U_STREAM, U_UNKNOWN };
void put(const void* p, hipStream_t s, Use use) noexcept {
  if (!p) return;
  State& S = state();
  std::lock_guard<std::mutex> g(S.mu);
  auto it = S.used.find(p);
  if (it == S.used.end()) {
    (void)hipFree(const_cast<void*>(p));
    return;
  }
  const int device = it->second.first;
  Block b = it->second.second;
  S.used.erase(it);
  // the per-thread handle names another stream in each thread: what this
  // thread's has done says nothing of the work another thread queued
  if (use == U_UNKNOWN || (use == U_STREAM && s == hipStreamPerThread)) {
    drop(b);  // hipFree waits for the device
    return;
  }
  // a stream that has run dry needs no event: most calls wait for their results
  // before they give their workspaces back (with an event each, a refinement
  // of 7 candidates took 646 us for 605, 16 subtomograms of 32^3 540 for 415)
  b.idle = use == U_NONE || hipStreamQuery(s) == hipSuccess;
  if (!b.idle) {
    (void)hipGetLastError();  // not ready
    if (!b.ev && hipEventCreateWithFlags(&b.ev, hipEventDisableTiming) != hipSuccess) b.ev = nullptr;
    if (!b.ev || hipEventRecord(b.ev, s) != hipSuccess) {
      (void)hipGetLastError();
      drop(b);
      return;
    }
  }
  try {
    keep(device, b);
  } catch (...) {
    drop(b);
  }
}

}  // namespace

void* device_malloc(size_t bytes) {
  State& S = state();
  int device = 0;
  TOMHIP_CHECK(hipGetDevice(&device));
  std::lock_guard<std::mutex> g(S.mu);
  return malloc_or_drop(S.dev[device], bytes);
}

void* work_get(size_t bytes, hipStream_t s) {
  State& S = state();
  const size_t want = rounded(bytes ? bytes : 1);
  int device = 0;
  TOMHIP_CHECK(hipGetDevice(&device));
  std::lock_guard<std::mutex> g(S.mu);
  Device& d = S.dev[device];
  // the smallest kept block that fits without wasting more than a quarter
  // (or a page), one that nothing uses first
  int best = -1;
  for (int i = 0; i < (int)d.kept.size(); ++i) {
    const Block& b = d.kept[i];
    if (b.size < want || b.size > want + want / 4 + 4096) continue;
    if (best < 0) {
      best = i;
      continue;
    }
    const Block& c = d.kept[best];
    if (b.idle != c.idle ? b.idle : b.size < c.size) best = i;
  }
  Block b;
  if (best >= 0) {
    b = d.kept[best];
    if (!b.idle && hipStreamWaitEvent(s, b.ev, 0) != hipSuccess) {
      (void)hipGetLastError();
      TOMHIP_CHECK(hipEventSynchronize(b.ev));
    }
    d.kept.erase(d.kept.begin() + best);
    d.bytes -= b.size;
  } else {
    b.p = malloc_or_drop(d, want);
    b.size = want;
  }
  try {
    S.used.emplace(b.p, std::make_pair(device, b));
  } catch (...) {
    drop(b);
    throw;
  }
  return b.p;
}

void work_put(const void* p, hipStream_t s) noexcept { put(p, s, U_STREAM); }
void work_put_all(std::initializer_list<const void*> ps) noexcept {
  const Use use = hipDeviceSynchronize() == hipSuccess ? U_NONE : U_UNKNOWN;
  if (use == U_UNKNOWN) (void)hipGetLastError();
  for (const void* p : ps) put(p, nullptr, use);
}

void work_trim(int device) {
  State& S = state();
  std::lock_guard<std::mutex> g(S.mu);
  drop_all(S.dev[device]);
}

void work_device_up(int device) {
  State& S = state();
  std::lock_guard<std::mutex> g(S.mu);
  ++S.dev[device].contexts;
}
void work_device_down(int device) noexcept {
  State& S = state();
  std::lock_guard<std::mutex> g(S.mu);
  Device& d = S.dev[device];
  if (--d.contexts == 0) drop_all(d);
}

}  // namespace tomhip
