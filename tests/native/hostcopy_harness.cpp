// Test harness: the host copies (channel_flow_amd/csrc/hostcopy.hip, over
// tests/native/hipstub) when their n-th allocation fails, a thread's start among
// them, run by tests/test_hostcopy_host.py.  Every copy has to be whole, and the
// pool's lanes have to be there again for the next one.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <new>
#include <vector>

#include "../../channel_flow_amd/csrc/hostcopy.hip"

static std::atomic<long> left{-1};  // allocations until one fails (-1: none does)

static void* take(std::size_t n) {
  if (left.load() >= 0 && left.fetch_sub(1) == 0) throw std::bad_alloc();
  if (void* p = std::malloc(n ? n : 1)) return p;
  throw std::bad_alloc();
}
void* operator new(std::size_t n) { return take(n); }
void* operator new[](std::size_t n) { return take(n); }
void operator delete(void* p) noexcept { std::free(p); }
void operator delete(void* p, std::size_t) noexcept { std::free(p); }
void operator delete[](void* p) noexcept { std::free(p); }
void operator delete[](void* p, std::size_t) noexcept { std::free(p); }

using namespace chf;

// a small array, one of less than a chunk more than a few, and a long one
static const std::size_t kBytes[3] = {1000, (std::size_t(7) << 20) + 13, std::size_t(45) << 20};

static int copy(Ctx& c, std::vector<char>* dev, std::vector<char>* host, bool to_host) {
  HostArray a[3];
  for (int i = 0; i < 3; ++i) a[i] = {dev[i].data(), host[i].data(), kBytes[i]};
  return (int)copy_arrays(c, a, 3, to_host);
}

// Lanes made for loading an array with one context alive, and with two.
static int lanes_for_load(Ctx& c, std::size_t bytes, int contexts) {
  std::vector<char> from(bytes, 7), to(bytes);
  const HostArray a[] = {{to.data(), from.data(), bytes}};
  for (int i = 0; i < contexts; ++i) hostcopy_retain();
  const bool ok = copy_arrays(c, a, 1, false) == hipSuccess && to == from;
  const int made = g_pool.devices[c.device].made;
  for (int i = 0; i < contexts; ++i) hostcopy_release();
  return ok ? made : -1;
}

// One array of a few chunks through a pool of its own: the streams made for it.
static int streams_for(Ctx& c, std::size_t bytes) {
  std::vector<char> from(bytes, 5), to(bytes);
  const HostArray a[] = {{from.data(), to.data(), bytes}};
  const int before = streams_made;
  hostcopy_retain();
  const bool ok = copy_arrays(c, a, 1, true) == hipSuccess && copy_arrays(c, a, 1, true) == hipSuccess && to == from;
  hostcopy_release();
  return ok ? streams_made - before : -1;
}

int main() {
  Ctx c;
  // a context of device 1, called with device 0 current
  (void)hipSetDevice(1);
  c.device = 1;
  (void)hipStreamCreateWithFlags(&c.stream, hipStreamNonBlocking);
  (void)hipStreamCreateWithFlags(&c.side, hipStreamNonBlocking);
  (void)hipSetDevice(0);
  std::printf("streams %d %d %d\n", streams_for(c, std::size_t(5) << 20), streams_for(c, std::size_t(12) << 20),
              streams_for(c, std::size_t(100) << 20));
  std::vector<char> from[3], to[3];
  for (int i = 0; i < 3; ++i) {
    from[i].resize(kBytes[i]);
    for (std::size_t k = 0; k < kBytes[i]; ++k) from[i][k] = (char)(k * 31 + (k >> 11) + i);
  }
  std::printf("lanes %d %d %d %d\n", lanes_for_load(c, std::size_t(3) << 20, 2), lanes_for_load(c, std::size_t(14) << 20, 1),
              lanes_for_load(c, std::size_t(14) << 20, 2), lanes_for_load(c, std::size_t(50) << 20, 1));
  for (int to_host = 0; to_host < 2; ++to_host)
    for (long n = 0;; ++n) {
      hostcopy_retain();  // a fresh pool each time
      bool hit = false;
      for (int again = 0; again < 2; ++again) {  // the second copy without a failure
        for (auto& t : to) t.assign(t.size(), 0);
        for (int i = 0; i < 3; ++i) to[i].resize(kBytes[i]);
        left = again ? -1 : n;
        const int rc = to_host ? copy(c, from, to, true) : copy(c, to, from, false);
        if (!again) hit = left.load() < 0;
        left = -1;
        for (int i = 0; i < 3; ++i)
          if (rc || to[i] != from[i] || current_device) return std::printf("%ld %d array %d: rc %d\n", n, again, i, rc), 1;
        if (again) {
          const int lanes = g_pool.devices[1].nidle;
          std::printf("%d %ld %d\n", to_host, n, lanes);
          std::fflush(stdout);
        }
      }
      hostcopy_release();
      if (!hit) break;  // n is past the last allocation
    }
  return 0;
}
