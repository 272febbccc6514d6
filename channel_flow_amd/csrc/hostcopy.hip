// Copies between device fields and the caller's pageable host arrays.
//
// A plain hipMemcpy of pageable memory moves about 10 GB/s here: one thread
// copies through the runtime's staging buffer, and a freshly allocated
// destination takes its page faults in that copy.  Here several threads move
// chunks, each through two pinned buffers of its own and on a stream of its own
// (the first two on the context's, which are idle then): while one buffer's transfer is in flight the other is copied to or from the
// caller's array, so the copies and page faults run in parallel with the link.
// Bound: the link (and, for a new destination, the page faults).  A state record
// at 256x193x256 (0.81 GB): read 61 -> 12.7 ms, loaded 23 -> 11.2 ms; one physical
// field at 512x257x512 (0.54 GB) 54.8 -> 12.1 ms, new pages every time.  Read rates
// with 4 / 6 / 8 lanes: 59 / 68 / 68 GB/s.
//
// The pinned buffers and streams are kept in a process-wide pool per device, at
// most kMaxLanes lanes (2 x kChunk bytes each); a lane belongs to one call at a
// time, and the pool is freed when the last context is destroyed.  A stream costs
// 0.5 ms to make and 0.6 to destroy, the buffers 0.2 and 0.1: with a stream in every
// lane a program that makes a context, loads, reads and destroys it paid up to 2 ms
// at the first copy and 4 at the end.  A copy itself
// allocates nothing but its threads: without memory it has fewer lanes or threads,
// or goes the plain way, and never throws.
#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>

#include "chf_internal.h"

namespace chf {

namespace {

constexpr size_t kChunk = size_t(2) << 20;
constexpr int kMaxLanes = 6;
// Smaller transfers go the plain way.  Loading, which meets no page faults, is as
// fast so up to about 40 MB while one context is alive: records of 13 MB 0.6 ms, through
// lanes 1.0; 43 MB 1.6 / 1.1; two fields into a new context, which makes its lanes
// then, 14 MB 0.7 / 1.3, 34 MB 1.6 / 2.8, 95 MB 6.4 / 5.1.  With several contexts the
// runtime's copy is slower: 14 MB into each of two 0.75, of three 2.2, of sixteen 4.6 ms,
// through lanes 1.2, 1.1, 0.7 (an ensemble of 24 loaded 93 / 19).
constexpr size_t kMinBytes = size_t(4) << 20, kMinLoadAlone = size_t(40) << 20;

struct Lane {
  hipStream_t stream = nullptr;  // made for a call's third lane on
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
  hipError_t e = hipSuccess;
  for (int b = 0; b < 2 && e == hipSuccess; ++b) {
    e = hipHostMalloc(&l.pin[b], kChunk, hipHostMallocDefault);
    if (e == hipSuccess) e = hipEventCreateWithFlags(&l.done[b], hipEventDisableTiming);
  }
  return e;
}

struct DeviceLanes {
  Lane idle[kMaxLanes];
  int nidle = 0, made = 0;
};

struct Pool {
  std::mutex mu;
  int users = 0;  // contexts alive
  std::map<int, DeviceLanes> devices;
} g_pool;

// Lanes of a context's device for one call, given back at its end.
struct Lanes {
  Lane lane[kMaxLanes];
  int n = 0;
  const int device;

  explicit Lanes(int dev) : device(dev) {}
  Lanes(const Lanes&) = delete;

  // An idle lane, with or without a stream of its own as wanted where there is one.
  static Lane pick(DeviceLanes& d, bool stream) {
    int k = d.nidle - 1;
    while (k > 0 && (d.idle[k].stream != nullptr) != stream) --k;
    std::swap(d.idle[k], d.idle[--d.nidle]);
    return d.idle[d.nidle];
  }

  // up to `want` (none if all are taken or cannot be made), from the third on with
  // streams of their own; made on the context's device, whichever is current
  void take(int want) {
    const DeviceScope here(device);
    if (!here.ok()) return;
    std::lock_guard<std::mutex> lock(g_pool.mu);
    DeviceLanes* d = nullptr;
    try {
      d = &g_pool.devices[device];
    } catch (...) {
      return;
    }
    while (n < want) {
      const bool own = n >= 2;
      Lane l;
      if (d->nidle > 0) {
        l = pick(*d, own);
      } else {
        if (d->made >= kMaxLanes) break;
        if (lane_make(l) != hipSuccess) {
          lane_free(l);
          (void)hipGetLastError();
          break;
        }
        ++d->made;
      }
      if (own && !l.stream && hipStreamCreateWithFlags(&l.stream, hipStreamNonBlocking) != hipSuccess) {
        l.stream = nullptr;
        (void)hipGetLastError();
        d->idle[d->nidle++] = l;
        break;
      }
      lane[n++] = l;
    }
  }

  ~Lanes() {
    if (n == 0) return;
    std::lock_guard<std::mutex> lock(g_pool.mu);
    DeviceLanes& d = g_pool.devices.find(device)->second;
    for (int i = 0; i < n; ++i) d.idle[d.nidle++] = lane[i];
  }
};

struct Job {
  char* dev;
  char* host;
  size_t bytes;
};

// The chunks of the arrays that go through the lanes, in turn.
struct Jobs {
  const HostArray* arrays;
  int count;

  static size_t chunks(const HostArray& a) { return a.bytes < kChunk ? 0 : (a.bytes + kChunk - 1) / kChunk; }
  bool get(size_t i, Job& j) const {
    for (int k = 0; k < count; ++k) {
      const size_t n = chunks(arrays[k]), o = i * kChunk;
      if (i < n) {
        j = {(char*)arrays[k].dev + o, (char*)arrays[k].host + o, std::min(kChunk, arrays[k].bytes - o)};
        return true;
      }
      i -= n;
    }
    return false;
  }
};

hipError_t run_lane(Lane& l, hipStream_t stream, const Jobs& jobs, std::atomic<size_t>& next, bool to_host) {
  Job held[2] = {};  // bytes: of the transfer in flight into the buffer, or 0
  bool used[2] = {false, false};
  hipError_t e = hipSuccess;
  auto finish = [&](int b) {
    if (!held[b].bytes) return;
    e = hipEventSynchronize(l.done[b]);
    if (e == hipSuccess) std::memcpy(held[b].host, l.pin[b], held[b].bytes);
    held[b].bytes = 0;
  };
  int b = 0;
  Job j;
  for (; e == hipSuccess && jobs.get(next++, j); b ^= 1) {
    if (to_host) {
      e = hipMemcpyAsync(l.pin[b], j.dev, j.bytes, hipMemcpyDeviceToHost, stream);
      if (e == hipSuccess) e = hipEventRecord(l.done[b], stream);
      if (e != hipSuccess) break;
      held[b] = j;
      finish(b ^ 1);
    } else {
      if (used[b]) e = hipEventSynchronize(l.done[b]);
      if (e != hipSuccess) break;
      std::memcpy(l.pin[b], j.host, j.bytes);
      e = hipMemcpyAsync(j.dev, l.pin[b], j.bytes, hipMemcpyHostToDevice, stream);
      if (e == hipSuccess) e = hipEventRecord(l.done[b], stream);
      used[b] = true;
    }
  }
  if (e == hipSuccess) finish(b ^ 1);
  const hipError_t s = hipStreamSynchronize(stream);  // the buffers are free again
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
  for (auto& d : g_pool.devices) {
    for (int i = 0; i < d.second.nidle; ++i) lane_free(d.second.idle[i]);
    d.second.made -= d.second.nidle;
    d.second.nidle = 0;
  }
}

// Bytes from which a copy goes through lanes.
static size_t lanes_from(bool to_host) {
  std::lock_guard<std::mutex> lock(g_pool.mu);
  return to_host || g_pool.users > 1 ? kMinBytes : kMinLoadAlone;
}

hipError_t copy_arrays(Ctx& c, const HostArray* arrays, int count, bool to_host) {
  size_t total = 0;
  for (int k = 0; k < count; ++k)
    if (arrays[k].bytes >= kChunk) total += arrays[k].bytes;
  Lanes lanes(c.device);
  if (total >= lanes_from(to_host)) lanes.take((int)std::min<size_t>(kMaxLanes, total / (4 * kChunk) + 1));
  for (int k = 0; k < count; ++k) {
    const HostArray& a = arrays[k];
    if (lanes.n > 0 && a.bytes >= kChunk) continue;
    const hipError_t e = to_host ? hipMemcpyAsync(a.host, a.dev, a.bytes, hipMemcpyDeviceToHost, c.stream)
                                 : hipMemcpyAsync(a.dev, a.host, a.bytes, hipMemcpyHostToDevice, c.stream);
    if (e != hipSuccess) return e;
  }
  // the lanes' streams start after the work queued on the context's streams (the
  // side stream's is joined to the first's), and what is queued there next starts
  // after them
  hipError_t e = hipStreamSynchronize(c.stream);
  if (e != hipSuccess || lanes.n == 0) return e;
  const Jobs jobs{arrays, count};
  std::atomic<size_t> next{0};
  hipError_t err[kMaxLanes] = {};
  auto lane = [&](int i) {
    if (i) err[i] = hipSetDevice(c.device);  // a helper thread of this call
    hipStream_t stream = i == 0 ? c.stream : i == 1 ? c.side : lanes.lane[i].stream;
    if (err[i] == hipSuccess) err[i] = run_lane(lanes.lane[i], stream, jobs, next, to_host);
  };
  std::thread threads[kMaxLanes];
  for (int i = 1; i < lanes.n; ++i) {
    try {
      threads[i] = std::thread(lane, i);
    } catch (...) {
      break;  // fewer threads: the others take the remaining chunks
    }
  }
  lane(0);
  for (std::thread& t : threads)
    if (t.joinable()) t.join();
  for (hipError_t x : err)
    if (e == hipSuccess) e = x;
  return e;
}

}  // namespace chf
