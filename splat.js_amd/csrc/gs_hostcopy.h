// gs_hostcopy.h — device results into the caller's pageable memory.
//
// A copy to pageable memory runs at the rate at which one CPU thread copies
// and, for a fresh array, faults its pages in: 13 GB/s for a 33 MB image.
// Here kernels fill the blocks of a small pinned ring and a few threads
// copy block after block to the caller while the next ones arrive. Renders
// into fresh arrays against a plain copy: 64x64 132 -> 65 us, 480x360 290 ->
// 211, 1280x720 1.16 -> 0.65 ms, 1920x1080 2.6 -> 1.3; a trainer's first one
// 530 -> 230 us at 480x360, 1.25 -> 0.75 ms at 1280x720. Reads of 73 MB of
// Gaussians 17.9 -> 2.4 ms (those also pinned and freed their whole size on
// each call).
//
// Kernels, not the copy engine: a copy of its own behind a kernel starts up to
// 130 us late. Through it the ring took 280 us for a 320x240 view that takes
// 110-130 now (163-290 by a plain copy), and 430 instead of 210 at 480x360.
// Four threads: their stacks stay in the C library's cache from call to call,
// which keeps 40 MB (five of 8 MB). With six or eight a trainer's first render
// took 1.1-2.4 ms at 1280x720 and 3.0-4.0 at 1920x1080 instead of 0.9 and 1.7;
// later ones are within 5%. Blocks of 1 MB are within 10% of 2 MB, 0.5 MB cost
// 20% more at 1920x1080. The first render of a program, 1920x1080: 14.9 ms by a
// plain copy, 9.0 by the copy engine and eight threads, 3.1 now.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

namespace gs {

// Pinned blocks of one trainer, as many as its largest read so far needs, at
// most kSlots, freed with it (pinning takes 70 us per MB). A trainer's calls
// do not overlap, so one reader uses them at a time.
struct HostRing {
  static constexpr int kSlots = 8;
  static constexpr size_t kSlotBytes = size_t(2) << 20;
  static constexpr int kWorkers = 4;
  char* buf = nullptr;
  size_t have = 0;
  hipEvent_t ev[kSlots] = {};   // slot filled

  // room for `slots` slots of `bytes` each; nothing may be in flight
  hipError_t ensure(int slots, size_t bytes) {
    hipError_t e = hipSuccess;
    const size_t need = slots * bytes;
    if (need > have) {
      const size_t all = kSlots * kSlotBytes, size = std::min(all, std::max(need, 2 * have));
      if (buf) (void)hipHostFree(buf);
      buf = nullptr;
      have = 0;
      e = hipHostMalloc((void**)&buf, size, hipHostMallocDefault);
      if (e != hipSuccess) buf = nullptr;
      else have = size;
    }
    for (int k = 0; k < slots && e == hipSuccess; k++)
      if (!ev[k]) e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    return e;
  }
  void release() {
    for (hipEvent_t& e : ev) {
      if (e) (void)hipEventDestroy(e);
      e = nullptr;
    }
    if (buf) (void)hipHostFree(buf);
    buf = nullptr;
    have = 0;
  }
};

// `count` blocks of at most `bytes` (<= kSlotBytes) through the ring:
// fill(k, slot) enqueues on st what writes block k into the pinned slot,
// take(k, slot) copies it to the caller on any thread. Returns when all have
// been taken, or with an error once nothing is being written or taken. Where
// the pinned memory cannot be had the call is plain(error)'s.
template <typename Fill, typename Take, typename Plain>
hipError_t ring_copy(HostRing& ring, hipStream_t st, int count, size_t bytes, Fill fill, Take take, Plain plain) {
  if (count <= 0) return hipSuccess;
  const size_t stride = std::min((bytes + 4095) / 4096 * 4096, HostRing::kSlotBytes);
  hipError_t e = ring.ensure(std::min(count, HostRing::kSlots), stride);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    return plain(e);
  }
  const auto slot = [&](int k) { return ring.buf + (size_t)(k % HostRing::kSlots) * stride; };
  std::mutex m;
  std::condition_variable some, freed;
  int arrived = 0, next = 0;             // blocks in the ring, the next one to take
  bool stop = false;
  bool busy[HostRing::kSlots] = {};      // the slot's block has not been taken yet
  // takes blocks until none is left; the caller's thread joins in at the end
  const auto work = [&] {
    std::unique_lock<std::mutex> l(m);
    for (;;) {
      some.wait(l, [&] { return stop || next >= count || next < arrived; });
      if (stop || next >= count) return;
      const int k = next++;
      if (next >= count) some.notify_all();
      l.unlock();
      take(k, slot(k));
      l.lock();
      busy[k % HostRing::kSlots] = false;
      freed.notify_one();
    }
  };
  // a thread that cannot be started leaves its share to the others
  std::vector<std::thread> threads;
  const int hw = (int)std::thread::hardware_concurrency();
  const int workers = count < 3 ? 0 : std::min({HostRing::kWorkers, count - 1, hw > 1 ? hw - 1 : 0});
  try {
    threads.reserve((size_t)workers);
    for (int t = 0; t < workers; t++) threads.emplace_back(work);
  } catch (...) {
  }
  int sent = 0;
  for (int k = 0; k < count && e == hipSuccess; k++) {
    for (; sent < count && e == hipSuccess; sent++) {
      const int s = sent % HostRing::kSlots;
      {
        std::unique_lock<std::mutex> l(m);
        if (busy[s]) {
          if (sent > k) break;             // others are on their way
          freed.wait(l, [&] { return !busy[s]; });
        }
        busy[s] = true;
      }
      e = fill(sent, slot(sent));
      if (e == hipSuccess) e = hipEventRecord(ring.ev[s], st);
    }
    if (e == hipSuccess) e = hipEventSynchronize(ring.ev[k % HostRing::kSlots]);
    if (e != hipSuccess) break;
    if (threads.empty()) {
      take(k, slot(k));
      busy[k % HostRing::kSlots] = false;
      next = k + 1;
      continue;
    }
    std::lock_guard<std::mutex> l(m);
    arrived = k + 1;
    some.notify_one();
  }
  if (e != hipSuccess) {
    std::lock_guard<std::mutex> l(m);
    stop = true;
    some.notify_all();
  }
  if (!threads.empty()) work();
  for (std::thread& t : threads) t.join();
  if (e != hipSuccess) (void)hipStreamSynchronize(st);   // fills behind the failed one
  return e;
}

// Pinned statistics blocks with their events, shared by a trainer and the
// readbacks it started (which may outlive it and end on any thread). Keeps
// up to kKeep free ones.
struct StatPool {
  static constexpr size_t kKeep = 4;
  struct Block {
    double* stats = nullptr;
    hipEvent_t ev = nullptr;
  };
  const int device;
  const size_t bytes;
  std::mutex m;
  std::vector<Block> free;

  StatPool(int device, size_t bytes) : device(device), bytes(bytes) { free.reserve(kKeep); }
  ~StatPool() {
    (void)hipSetDevice(device);
    for (Block& b : free) destroy(b);
  }
  static void destroy(Block& b) {
    if (b.ev) (void)hipEventDestroy(b.ev);
    if (b.stats) (void)hipHostFree(b.stats);
    b = Block{};
  }
  hipError_t get(Block& b) {
    {
      std::lock_guard<std::mutex> l(m);
      if (!free.empty()) {
        b = free.back();
        free.pop_back();
        return hipSuccess;
      }
    }
    hipError_t e = hipEventCreateWithFlags(&b.ev, hipEventDisableTiming);
    if (e == hipSuccess) e = hipHostMalloc((void**)&b.stats, bytes, hipHostMallocDefault);
    if (e != hipSuccess) destroy(b);
    return e;
  }
  // the block's event has passed
  void put(Block& b) {
    {
      std::lock_guard<std::mutex> l(m);
      if (free.size() < kKeep) {
        free.push_back(b);
        b = Block{};
        return;
      }
    }
    destroy(b);
  }
};

}  // namespace gs
