// Copies between device fields and the caller's pageable host arrays.
//
// A plain hipMemcpy of pageable memory moves about 10 GB/s here: one thread
// copies through the runtime's staging buffer, and a freshly allocated
// destination takes its page faults in that copy.  Here several threads move
// chunks, each through two pinned buffers of its own and on a stream of its own:
// while one buffer's transfer is in flight the other is copied to or from the
// caller's array, so the copies and page faults run in parallel with the link.
// Bound: the link (and, for a new destination, the page faults).  A state record
// at 256x193x256 (0.81 GB): read 61 -> 12.7 ms, loaded 23 -> 11.2 ms; one physical
// field at 512x257x512 (0.54 GB) 54.8 -> 12.1 ms, new pages every time.  Read rates
// with 4 / 6 / 8 lanes: 59 / 68 / 68 GB/s.
//
// The pinned buffers and streams are kept in a process-wide pool per device, at
// most kMaxLanes lanes (2 x kChunk bytes each); a lane belongs to one call at a
// time, and the pool is freed when the last context is destroyed.
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "chf_internal.h"

namespace chf {

namespace {

constexpr size_t kChunk = size_t(2) << 20;
constexpr int kMaxLanes = 6;
constexpr size_t kMinBytes = size_t(4) << 20;  // smaller transfers go the plain way

struct Lane {
  hipStream_t stream = nullptr;
  void* pin[2] = {nullptr, nullptr};
  hipEvent_t done[2] = {nullptr, nullptr};
};

void lane_free(Lane& l) {
  for (int b = 0; b < 2; ++b) {
    if (l.pin[b]) (void)hipHostFree(l.pin[b]);
    if (l.done[b]) (void)hipEventDestroy(l.done[b]);
  }
  if (l.stream) (void)hipStreamDestroy(l.stream);
}

hipError_t lane_make(Lane& l) {
  hipError_t e = hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking);
  for (int b = 0; b < 2 && e == hipSuccess; ++b) {
    e = hipHostMalloc(&l.pin[b], kChunk, hipHostMallocDefault);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&l.done[b], hipEventDisableTiming);
  }
  return e;
}

struct Pool {
  std::mutex mu;
  int users = 0;                          // contexts alive
  std::map<int, std::vector<Lane>> idle;  // by device
  std::map<int, int> made;
} g_pool;

// Up to `want` lanes of the current device (none if all are taken or cannot be made).
std::vector<Lane> take_lanes(int device, int want) {
  std::lock_guard<std::mutex> lock(g_pool.mu);
  std::vector<Lane>& idle = g_pool.idle[device];
  int& made = g_pool.made[device];
  std::vector<Lane> got;
  while ((int)got.size() < want) {
    if (!idle.empty()) {
      got.push_back(idle.back());
      idle.pop_back();
      continue;
    }
    if (made >= kMaxLanes) break;
    Lane l;
    if (lane_make(l) != hipSuccess) {
      lane_free(l);
      (void)hipGetLastError();
      break;
    }
    ++made;
    got.push_back(l);
  }
  return got;
}

void give_lanes(int device, const std::vector<Lane>& lanes) {
  std::lock_guard<std::mutex> lock(g_pool.mu);
  for (const Lane& l : lanes) g_pool.idle[device].push_back(l);
}

struct Job {
  char* dev;
  char* host;
  size_t bytes;
};

hipError_t run_lane(Lane& l, const std::vector<Job>& jobs, std::atomic<size_t>& next, bool to_host) {
  const Job* held[2] = {nullptr, nullptr};
  bool used[2] = {false, false};
  hipError_t e = hipSuccess;
  auto finish = [&](int b) {
    if (!held[b]) return;
    e = hipEventSynchronize(l.done[b]);
    if (e == hipSuccess) std::memcpy(held[b]->host, l.pin[b], held[b]->bytes);
    held[b] = nullptr;
  };
  int b = 0;
  for (size_t i = next++; i < jobs.size() && e == hipSuccess; i = next++, b ^= 1) {
    const Job& j = jobs[i];
    if (to_host) {
      e = hipMemcpyAsync(l.pin[b], j.dev, j.bytes, hipMemcpyDeviceToHost, l.stream);
      if (e == hipSuccess) e = hipEventRecord(l.done[b], l.stream);
      if (e != hipSuccess) break;
      held[b] = &j;
      finish(b ^ 1);
    } else {
      if (used[b]) e = hipEventSynchronize(l.done[b]);
      if (e != hipSuccess) break;
      std::memcpy(l.pin[b], j.host, j.bytes);
      e = hipMemcpyAsync(j.dev, l.pin[b], j.bytes, hipMemcpyHostToDevice, l.stream);
      if (e == hipSuccess) e = hipEventRecord(l.done[b], l.stream);
      used[b] = true;
    }
  }
  if (e == hipSuccess) finish(b ^ 1);
  const hipError_t s = hipStreamSynchronize(l.stream);  // the buffers are free again
  return e != hipSuccess ? e : s;
}

}  // namespace

void hostcopy_retain() {
  std::lock_guard<std::mutex> lock(g_pool.mu);
  ++g_pool.users;
}

void hostcopy_release() {
  std::lock_guard<std::mutex> lock(g_pool.mu);
  if (--g_pool.users > 0) return;
  for (auto& d : g_pool.idle) {
    g_pool.made[d.first] -= (int)d.second.size();
    for (Lane& l : d.second) lane_free(l);
    d.second.clear();
  }
}

hipError_t copy_arrays(Ctx& c, const std::vector<HostArray>& arrays, bool to_host) {
  size_t total = 0;
  std::vector<Job> jobs;
  for (const HostArray& a : arrays)
    if (a.bytes >= kChunk) total += a.bytes;
  std::vector<Lane> lanes;
  if (total >= kMinBytes) lanes = take_lanes(c.device, std::min<int>(kMaxLanes, (int)(total / (4 * kChunk)) + 1));
  for (const HostArray& a : arrays) {
    if (lanes.empty() || a.bytes < kChunk) {
      const hipError_t e = to_host ? hipMemcpyAsync(a.host, a.dev, a.bytes, hipMemcpyDeviceToHost, c.stream)
                                   : hipMemcpyAsync(a.dev, a.host, a.bytes, hipMemcpyHostToDevice, c.stream);
      if (e != hipSuccess) {
        give_lanes(c.device, lanes);
        return e;
      }
      continue;
    }
    for (size_t o = 0; o < a.bytes; o += kChunk)
      jobs.push_back({(char*)a.dev + o, (char*)a.host + o, std::min(kChunk, a.bytes - o)});
  }
  // the lanes' streams start after the work queued on the context's stream, and
  // what is queued there next starts after them
  hipError_t e = hipStreamSynchronize(c.stream);
  if (e == hipSuccess && !lanes.empty()) {
    std::atomic<size_t> next{0};
    std::vector<hipError_t> err(lanes.size(), hipSuccess);
    auto lane = [&](size_t i) {
      if (i) err[i] = hipSetDevice(c.device);  // the caller's thread has it current
      if (err[i] == hipSuccess) err[i] = run_lane(lanes[i], jobs, next, to_host);
    };
    std::vector<std::thread> threads;
    threads.reserve(lanes.size());
    try {
      for (size_t i = 1; i < lanes.size(); ++i) threads.emplace_back(lane, i);
    } catch (const std::system_error&) {
      // fewer threads: the others take the remaining chunks
    }
    lane(0);
    for (std::thread& t : threads) t.join();
    for (hipError_t x : err)
      if (e == hipSuccess) e = x;
  }
  give_lanes(c.device, lanes);
  return e;
}

}  // namespace chf
