// Device memory of the library's buffers.
//
// Building a plan and its first reconstruction take some 60 buffers, and
// hipMalloc / hipFree of them cost as much as the kernels: 8.7 of 24.4 ms at
// 128^3 (18.2 ms with the blocks passed on; 21.0 to 21.7 when all go back with the last
// context).  So a released block waits here for the next request of about its size.
//
// hipFree waits for the device; a block given up here may still be in use on
// some stream, so it is `pending` until one of the pending blocks -- the
// smallest -- goes back to the driver, when a request could be served by a
// pending block only: one wait for all that are pending.  (hipFree, since a
// device synchronisation would break a graph capture in progress in another
// thread.)  Where that fails, the request goes to the driver.  At most kBound
// bytes wait; a block past it goes back at once, and all do when the driver is
// out of memory, or on device_release_unused().
#include <map>
#include <mutex>

#include "devpool.hpp"

namespace omni3d {

namespace {

constexpr size_t kBound = (size_t)2 << 30;  // under a hundredth of the card's memory

struct Pool {
  std::mutex wait;  // held (before mu) while blocks are out of the lists to be waited for
  std::mutex mu;
  std::multimap<size_t, void*> ready, pending;  // by size
};

constexpr int kDevices = 16;
std::mutex g_mu;       // the total
size_t g_unused = 0;

// (never destroyed: buffers of static storage may outlive any other static)
Pool& pool(int dev) {
  static Pool* p = new Pool[kDevices];
  return p[dev];
}

// whole pages, whole 2 MiB fragments for large blocks
size_t rounded(size_t bytes) {
  const size_t g = bytes < ((size_t)2 << 20) ? (size_t)4096 : (size_t)2 << 20;
  return (bytes + g - 1) / g * g;
}

// the smallest block that wastes at most a quarter
bool fits(const std::multimap<size_t, void*>& m, size_t need) {
  const auto it = m.lower_bound(need);
  return it != m.end() && it->first <= need + need / 4;
}
void* take(std::multimap<size_t, void*>* m, size_t need, size_t* cap) {
  if (!fits(*m, need)) return nullptr;
  const auto it = m->lower_bound(need);
  void* p = it->second;
  *cap = it->first;
  m->erase(it);
  return p;
}

void count(size_t cap, bool add) {
  std::lock_guard<std::mutex> lock(g_mu);
  g_unused = add ? g_unused + cap : g_unused - cap;
}

size_t give_back(int dev) {
  std::multimap<size_t, void*> all;
  {
    // (blocks another thread waits for come back to the lists first)
    Pool& q = pool(dev);
    std::lock_guard<std::mutex> held(q.wait);
    std::lock_guard<std::mutex> lock(q.mu);
    all.swap(q.ready);
    all.merge(q.pending);
  }
  size_t bytes = 0;
  for (const auto& b : all) {
    (void)hipFree(b.second);  // (waits for the device)
    count(b.first, false);
    bytes += b.first;
  }
  return bytes;
}

// A pending block, after one of the others went back to the driver.
void* take_after_wait(Pool& q, size_t need, size_t* cap) {
  std::lock_guard<std::mutex> held(q.wait);
  std::multimap<size_t, void*> waited;
  {
    std::lock_guard<std::mutex> lock(q.mu);
    if (void* p = take(&q.ready, need, cap)) return p;
    if (!fits(q.pending, need)) return nullptr;
    waited.swap(q.pending);
  }
  auto fence = waited.begin();
  if (fence->first >= need) ++fence;
  const bool idle = fence != waited.end() && hipFree(fence->second) == hipSuccess;
  if (idle) {
    count(fence->first, false);
    waited.erase(fence);
  }
  std::lock_guard<std::mutex> lock(q.mu);
  (idle ? q.ready : q.pending).merge(waited);
  return idle ? take(&q.ready, need, cap) : nullptr;
}

}  // namespace

hipError_t device_alloc(void** p, size_t bytes, size_t* cap, int* dev) {
  *p = nullptr;
  hipError_t e = hipGetDevice(dev);
  if (e != hipSuccess) return e;
  const size_t need = rounded(bytes ? bytes : 1);
  if (*dev < kDevices) {
    Pool& q = pool(*dev);
    bool fence = false;
    {
      std::lock_guard<std::mutex> lock(q.mu);
      *p = take(&q.ready, need, cap);
      fence = !*p && fits(q.pending, need);
    }
    if (fence) *p = take_after_wait(q, need, cap);
    if (*p) {
      count(*cap, false);
      return hipSuccess;
    }
  }
  *cap = need;
  e = hipMalloc(p, need);
  if (e == hipErrorOutOfMemory && *dev < kDevices && give_back(*dev) > 0) {
    (void)hipGetLastError();
    e = hipMalloc(p, need);
  }
  if (e != hipSuccess) *p = nullptr;
  return e;
}

void device_free(void* p, size_t cap, int dev) {
  if (!p) return;
  bool keep = dev >= 0 && dev < kDevices;
  if (keep) {
    std::lock_guard<std::mutex> lock(g_mu);
    keep = g_unused + cap <= kBound;
    if (keep) g_unused += cap;
  }
  if (!keep) {
    (void)hipFree(p);
    return;
  }
  try {
    Pool& q = pool(dev);
    std::lock_guard<std::mutex> lock(q.mu);
    q.pending.emplace(cap, p);
  } catch (...) {  // (no host memory for the entry)
    count(cap, false);
    (void)hipFree(p);
  }
}

size_t device_release_unused() {
  size_t bytes = 0;
  for (int d = 0; d < kDevices; d++) bytes += give_back(d);
  return bytes;
}

}  // namespace omni3d
