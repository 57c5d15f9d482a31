// Device memory pools (declared in common.hpp).
#include <algorithm>
#include <map>
#include <new>

#include "common.hpp"

namespace sucem {

namespace {

// every pool that may hold unused blocks (never destroyed: buffers may outlive main)
struct PoolList {
  std::mutex mu;
  std::vector<std::weak_ptr<MemPool>> all;
};
PoolList& pool_list() {
  static PoolList* l = new PoolList();
  return *l;
}

// Sizes are rounded up by at most an eighth (4 KB and more; below that to 512 bytes), so that
// buffers of slightly different meshes share blocks.  A block that no pool can keep is not
// rounded: the largest matrices (17.3 GB of FP64 values on a cavity of 120 x 60 x 90 boxes)
// would only lose memory by it.
size_t block_size(size_t bytes) {
  if (bytes > MemPool::kMax) return bytes;
  size_t step = 512;
  while (step * 16 <= bytes) step *= 2;
  return (bytes + step - 1) / step * step;
}

}  // namespace

std::shared_ptr<MemPool>& current_pool() {
  static thread_local std::shared_ptr<MemPool> p;
  return p;
}

std::shared_ptr<MemPool> new_pool() {
  auto p = std::make_shared<MemPool>();
  PoolList& l = pool_list();
  std::lock_guard<std::mutex> hold(l.mu);
  l.all.erase(std::remove_if(l.all.begin(), l.all.end(), [](auto& w) { return w.expired(); }),
              l.all.end());
  l.all.push_back(p);
  return p;
}

size_t pools_unused(int device) {
  PoolList& l = pool_list();
  std::lock_guard<std::mutex> hold(l.mu);
  size_t n = 0;
  for (auto& w : l.all)
    if (auto q = w.lock())
      if (q->device == device) n += q->unused();
  return n;
}

void* device_alloc(size_t bytes) {
  void* p = nullptr;
  if (hipMalloc(&p, bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  std::vector<std::shared_ptr<MemPool>> pools;
  {
    PoolList& l = pool_list();
    std::lock_guard<std::mutex> hold(l.mu);
    for (auto& w : l.all)
      if (auto q = w.lock()) pools.push_back(q);
  }
  for (auto& q : pools) q->trim();
  SUCEM_HIP(hipMalloc(&p, bytes));
  return p;
}

bool device_free(void* p) {
  if (hipFree(p) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

DeviceWait::DeviceWait() : before_(bypass_pools()) {
  void* p = nullptr;
  if (hipMalloc(&p, 256) != hipSuccess) (void)hipGetLastError();
  if (!p || !device_free(p)) bypass_pools() = true;
}

bool& DeviceWait::bypass_pools() {
  static thread_local bool b = false;
  return b;
}

MemPool::~MemPool() { trim(); }

void* MemPool::take(size_t bytes, size_t& got) {
  const size_t want = block_size(bytes);
  {
    std::lock_guard<std::mutex> hold(mu_);
    auto it = free_.lower_bound(want);
    if (it != free_.end() && it->first <= std::max(want, bytes + bytes / 8)) {
      void* p = it->second;
      got = it->first;
      unused_ -= got;
      free_.erase(it);
      return p;
    }
  }
  try {
    void* p = device_alloc(want);
    got = want;
    return p;
  } catch (const Error&) {   // a nearly full device may still have the bytes themselves
    (void)hipGetLastError();
    if (want == bytes) throw;
  }
  void* p = device_alloc(bytes);
  got = bytes;
  return p;
}

void MemPool::put(void* p, size_t size) {
  {
    std::lock_guard<std::mutex> hold(mu_);
    if (!closed_ && unused_ + size <= kMax) {
      try {
        free_.emplace(size, p);
        unused_ += size;
        return;
      } catch (const std::bad_alloc&) {   // (destructors call this) back to the device
      }
    }
  }
  (void)device_free(p);
}

void MemPool::trim() {
  std::multimap<size_t, void*> old;
  {
    std::lock_guard<std::mutex> hold(mu_);
    old.swap(free_);
    unused_ = 0;
  }
  for (auto& e : old) (void)device_free(e.second);   // waits for the work that may still use it
}

size_t MemPool::unused() {
  std::lock_guard<std::mutex> hold(mu_);
  return unused_;
}

void MemPool::close() {
  {
    std::lock_guard<std::mutex> hold(mu_);
    closed_ = true;
  }
  trim();
}

}  // namespace sucem
