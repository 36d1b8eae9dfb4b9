// The device-memory pool (csrc/devpool.cpp) over a counting allocator in place
// of the driver's: no GPU.  argv[1] names the check; 0 is a pass.
#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdio>
#include <cstring>
#include <functional>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

#include "devpool.hpp"

using omni3d::device_alloc;
using omni3d::device_free;
using omni3d::device_release_unused;

namespace {

std::mutex mu;
std::map<void*, size_t> live;
size_t in_use = 0, limit = (size_t)-1;
uintptr_t next_address = 1 << 20;
std::vector<size_t> freed;                 // sizes, in order
std::function<void(size_t)> on_free;       // before a block goes
std::atomic<int> refused{0};

struct Block {
  void* p = nullptr;
  size_t cap = 0;
  int dev = 0;
};
hipError_t get(Block* b, size_t bytes) { return device_alloc(&b->p, bytes, &b->cap, &b->dev); }
void put(const Block& b) { device_free(b.p, b.cap, b.dev); }

int fails = 0;
#define EXPECT(c) \
  do { \
    if (!(c)) { \
      fails++; \
      std::printf("line %d: %s\n", __LINE__, #c); \
    } \
  } while (0)

constexpr size_t kMiB = (size_t)1 << 20, kGiB = (size_t)1 << 30;

// A released block serves again only after a block went back to the driver
// (whose free waits for the device), and the smallest one goes.
void reuse() {
  Block a, b, c;
  EXPECT(get(&a, 8 * kMiB) == hipSuccess && get(&b, 2 * kMiB) == hipSuccess);
  put(a);
  put(b);
  EXPECT(freed.empty() && in_use == 10 * kMiB);
  EXPECT(get(&c, 7 * kMiB) == hipSuccess);
  EXPECT(c.p == a.p && c.cap == 8 * kMiB);
  EXPECT(freed.size() == 1 && freed[0] == 2 * kMiB);
  // a lone waiting block has no other to wait by, and a quarter is the most
  // that a request may waste
  put(c);
  Block d, e;
  EXPECT(get(&d, 8 * kMiB) == hipSuccess && d.p != a.p && freed.size() == 1);
  put(d);
  EXPECT(get(&e, 6 * kMiB) == hipSuccess && e.cap == 6 * kMiB);
  put(e);
  EXPECT(device_release_unused() == 22 * kMiB && in_use == 0);
}

// At most 2 GiB wait; a block past that goes back at once.
void bound() {
  std::vector<Block> b(24);
  for (auto& x : b) EXPECT(get(&x, 100 * kMiB) == hipSuccess);
  for (auto& x : b) put(x);
  EXPECT(in_use <= 2 * kGiB && in_use + 100 * kMiB > 2 * kGiB);
  EXPECT(freed.size() == 4);
  Block big;
  EXPECT(get(&big, 3 * kGiB) == hipSuccess);
  put(big);
  EXPECT(freed.size() == 5 && freed.back() == 3 * kGiB);
  EXPECT(device_release_unused() == 20 * 100 * kMiB && in_use == 0);
  EXPECT(device_release_unused() == 0);
}

// What waits goes back before a request is refused.
void out_of_memory() {
  limit = 100 * kMiB;
  Block a, b, c;
  EXPECT(get(&a, 60 * kMiB) == hipSuccess);
  put(a);
  EXPECT(get(&b, 90 * kMiB) == hipSuccess && in_use == 90 * kMiB);
  EXPECT(get(&c, 20 * kMiB) == hipErrorOutOfMemory && c.p == nullptr);
  put(b);
  EXPECT(get(&c, 20 * kMiB) == hipSuccess);
  put(c);
  (void)device_release_unused();
  EXPECT(in_use == 0);
}

// The same while another thread waits by one of the blocks: those are not
// out of reach meanwhile.
void out_of_memory_beside_a_wait() {
  limit = 100 * kMiB;
  Block s, b1, b2, mine, other;
  EXPECT(get(&s, kMiB) == hipSuccess && get(&b1, 40 * kMiB) == hipSuccess &&
         get(&b2, 40 * kMiB) == hipSuccess);
  put(s);
  put(b1);
  put(b2);
  std::atomic<bool> waiting{false};
  on_free = [&](size_t bytes) {
    if (bytes != s.cap) return;
    waiting = true;
    for (int i = 0; i < 5000 && refused == 0; i++)
      std::this_thread::sleep_for(std::chrono::milliseconds(1));
    std::this_thread::sleep_for(std::chrono::milliseconds(200));
  };
  std::thread t([&] { EXPECT(get(&other, 40 * kMiB) == hipSuccess); });
  while (!waiting) std::this_thread::yield();
  EXPECT(get(&mine, 50 * kMiB) == hipSuccess);
  t.join();
  EXPECT(other.p == b1.p || other.p == b2.p);
  put(mine);
  put(other);
  (void)device_release_unused();
  EXPECT(in_use == 0);
}

}  // namespace

extern "C" {

hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipGetLastError() { return hipSuccess; }
hipError_t hipMalloc(void** p, size_t bytes) {
  std::lock_guard<std::mutex> lock(mu);
  if (in_use + bytes > limit) {
    refused++;
    return hipErrorOutOfMemory;
  }
  *p = reinterpret_cast<void*>(next_address);
  next_address += bytes;
  live[*p] = bytes;
  in_use += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  size_t bytes;
  {
    std::lock_guard<std::mutex> lock(mu);
    const auto it = live.find(p);
    if (it == live.end()) {
      fails++;
      std::printf("freed twice or never allocated\n");
      return hipErrorInvalidValue;
    }
    bytes = it->second;
  }
  if (on_free) on_free(bytes);
  std::lock_guard<std::mutex> lock(mu);
  live.erase(p);
  in_use -= bytes;
  freed.push_back(bytes);
  return hipSuccess;
}

}  // extern "C"

int main(int argc, char** argv) {
  const std::map<std::string, void (*)()> checks = {
      {"reuse", reuse},
      {"bound", bound},
      {"out_of_memory", out_of_memory},
      {"out_of_memory_beside_a_wait", out_of_memory_beside_a_wait},
  };
  const auto it = argc > 1 ? checks.find(argv[1]) : checks.end();
  if (it == checks.end()) return 2;
  it->second();
  return fails ? 1 : 0;
}
