// Results to host memory.
//
// A copy into pageable memory goes through the runtime's own staging on one
// thread, which also takes the page faults of an array the caller has just
// allocated: 16 MB of depths into a fresh array took 1.0 ms, three times the
// transfer.  CopyToHost stages it through page-locked slots instead: the copy
// engine fills a slot while a few threads move earlier ones out, faults
// included (BFS on Kronecker 22 with its depths: 1.37 ms before, 0.99 with it).
// Page-locked destinations and small results are copied straight.
//
// The slots are one per process (kSlots x kSlotBytes), taken by one copy at a
// time -- a copy that finds them taken uses the runtime's path -- and freed
// with the last handle.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "gg_common.h"

namespace gg {
namespace {

constexpr size_t kSlotBytes = size_t(1) << 20;
constexpr int kSlots = 8;
constexpr int kMovers = 4;                             // threads that empty slots
constexpr size_t kStagedBytes = 2 * kSlotBytes;        // smaller results go by the runtime

std::mutex g_slots_mu;          // held by the copy that uses the slots
std::mutex g_handles_mu;        // guards the count below
int64_t g_handles = 0;          // handles alive in the process
char* g_slots = nullptr;        // kSlots x kSlotBytes, page-locked

// Whether p is ordinary (pageable) host memory.
bool Pageable(const void* p) {
  hipPointerAttribute_t a;
  if (hipPointerGetAttributes(&a, p) != hipSuccess) {
    (void)hipGetLastError();  // the runtime does not know it
    return true;
  }
  return a.type == hipMemoryTypeUnregistered;
}

// The events that tell when a slot is filled, on the copy's device.
struct Events {
  hipEvent_t ev[kSlots] = {};
  Events() {
    for (hipEvent_t& e : ev) GG_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  ~Events() {
    for (hipEvent_t e : ev)
      if (e) (void)hipEventDestroy(e);
  }
};

// Chunk c (kSlotBytes each) passes through slot c % kSlots.  The calling
// thread issues the device copies, a slot's next one once its last chunk has
// been moved out; the movers take chunks in order.  False, with nothing done,
// if there is no thread to be had.
bool StagedCopy(gg_graph* g, char* host, const char* dev, size_t bytes) {
  Events events;
  const int64_t chunks = static_cast<int64_t>((bytes + kSlotBytes - 1) / kSlotBytes);
  std::atomic<int64_t> issued{0}, taken{0};
  std::atomic<int64_t> moved[kSlots];  // chunks moved out of each slot
  for (auto& m : moved) m = 0;
  std::atomic<int> error{hipSuccess};
  auto size_of = [&](int64_t c) { return std::min(kSlotBytes, bytes - static_cast<size_t>(c) * kSlotBytes); };
  auto mover = [&] {
    if (hipError_t e = hipSetDevice(g->device); e != hipSuccess) error = e;
    for (;;) {
      const int64_t c = taken.fetch_add(1);
      if (c >= chunks) return;
      while (issued.load(std::memory_order_acquire) <= c) {
        if (error.load() != hipSuccess) return;
        std::this_thread::yield();
      }
      const int s = static_cast<int>(c % kSlots);
      if (hipError_t e = hipEventSynchronize(events.ev[s]); e != hipSuccess) error = e;
      if (error.load() != hipSuccess) return;
      std::memcpy(host + c * kSlotBytes, g_slots + s * kSlotBytes, size_of(c));
      moved[s].fetch_add(1, std::memory_order_release);
    }
  };
  std::vector<std::thread> threads;
  threads.reserve(kMovers);
  auto finish = [&] {
    for (std::thread& t : threads) t.join();
  };
  try {
    try {
      for (int i = 0; i < kMovers; i++) threads.emplace_back(mover);
    } catch (const std::system_error&) {  // no more threads: with those there are
      if (threads.empty()) return false;
    }
    for (int64_t c = 0; c < chunks && error.load() == hipSuccess; c++) {
      const int s = static_cast<int>(c % kSlots);
      while (moved[s].load(std::memory_order_acquire) < c / kSlots && error.load() == hipSuccess)
        std::this_thread::yield();
      GG_HIP(hipMemcpyAsync(g_slots + s * kSlotBytes, dev + c * kSlotBytes, size_of(c), hipMemcpyDeviceToHost,
                            g->stream));
      GG_HIP(hipEventRecord(events.ev[s], g->stream));
      issued.store(c + 1, std::memory_order_release);
    }
  } catch (...) {
    error = hipErrorUnknown;
    finish();
    (void)hipStreamSynchronize(g->stream);  // no copy into the slots outlives this call
    throw;
  }
  finish();
  const hipError_t e = static_cast<hipError_t>(error.load());
  if (e != hipSuccess) {
    (void)hipStreamSynchronize(g->stream);
    GG_HIP(e);
  }
  return true;
}

}  // namespace

void CopyToHost(gg_graph* g, void* host, const void* dev, size_t bytes) {
  if (bytes >= kStagedBytes && Pageable(host)) {
    std::unique_lock<std::mutex> lk(g_slots_mu, std::try_to_lock);
    if (lk.owns_lock()) {
      if (!g_slots) {
        void* p = nullptr;
        if (hipHostMalloc(&p, kSlots * kSlotBytes, hipHostMallocPortable) != hipSuccess) {
          (void)hipGetLastError();  // no page-locked memory: the runtime's path
        } else {
          g_slots = static_cast<char*>(p);
        }
      }
      if (g_slots && StagedCopy(g, static_cast<char*>(host), static_cast<const char*>(dev), bytes)) return;
    }
  }
  GG_HIP(hipMemcpyAsync(host, dev, bytes, hipMemcpyDeviceToHost, g->stream));
  GG_HIP(hipStreamSynchronize(g->stream));
}

void HandleCreated() {
  std::lock_guard<std::mutex> lk(g_handles_mu);
  g_handles++;
}

void HandleFreed() {
  std::lock_guard<std::mutex> lk(g_handles_mu);
  if (--g_handles > 0) return;
  std::lock_guard<std::mutex> slots(g_slots_mu);
  if (g_slots) (void)hipHostFree(g_slots);
  g_slots = nullptr;
}

}  // namespace gg
