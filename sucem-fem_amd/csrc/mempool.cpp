// Device memory pools (declared in common.hpp).
#include <algorithm>
#include <atomic>
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

namespace {

std::vector<std::shared_ptr<MemPool>> live_pools() {
  PoolList& l = pool_list();
  std::lock_guard<std::mutex> hold(l.mu);
  std::vector<std::shared_ptr<MemPool>> pools;
  for (auto& w : l.all)
    if (auto q = w.lock()) pools.push_back(q);
  return pools;
}

// unused bytes of all pools of a device
std::atomic<size_t>& kept_on(int device) {
  static std::atomic<size_t> kept[256];
  return kept[(unsigned)device % 256];
}

}  // namespace

void trim_pools(int device) {
  for (auto& q : live_pools())
    if (q->device == device) q->trim();
}

void* device_alloc(size_t bytes) {
  void* p = nullptr;
  if (hipMalloc(&p, bytes) == hipSuccess) return p;
  (void)hipGetLastError();
  for (auto& q : live_pools()) q->trim();
  SUCEM_HIP(hipMalloc(&p, bytes));
  return p;
}

bool device_free(void* p) {
  const BesideCaptures beside;
  if (hipFree(p) == hipSuccess) return true;
  (void)hipGetLastError();
  return false;
}

DeviceWait::DeviceWait(hipStream_t owners) : before_(bypass_pools()) {
  const BesideCaptures beside;
  hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(owners, &cap) != hipSuccess ||
      (cap == hipStreamCaptureStatusNone && hipStreamSynchronize(owners) != hipSuccess))
    (void)hipGetLastError();
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
      void* p = it->second.p;
      got = it->first;
      unused_ -= got;
      kept_on(device) -= got;
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
  const auto now = Clock::now();
  try {   // (destructors call this: what cannot be kept goes back to the device)
    if (keep(p, size, now)) return;
    bool dropped = false;
    if (size <= kMax)
      for (auto& q : live_pools())
        if (q->device == device && q->drop_idle(now)) dropped = true;
    if (dropped && keep(p, size, now)) return;
  } catch (const std::bad_alloc&) {
  }
  (void)device_free(p);
}

bool MemPool::keep(void* p, size_t size, Clock::time_point now) {
  std::lock_guard<std::mutex> hold(mu_);
  if (closed_ || size > kMax || !look(now)) return false;
  if (kept_on(device).fetch_add(size) + size > limit_) {
    kept_on(device) -= size;
    return false;
  }
  try {
    free_.emplace(size, Block{p, now});
  } catch (const std::bad_alloc&) {
    kept_on(device) -= size;
    throw;
  }
  unused_ += size;
  return true;
}

bool MemPool::drop_idle(Clock::time_point now) {
  const auto old = now - std::chrono::milliseconds(kIdleMs);
  std::vector<void*> drop;
  {
    std::lock_guard<std::mutex> hold(mu_);
    if (oldest_ > old) return false;
    oldest_ = now;
    for (auto it = free_.begin(); it != free_.end();) {
      if (it->second.since > old) {
        oldest_ = std::min(oldest_, it->second.since);
        ++it;
        continue;
      }
      drop.push_back(it->second.p);
      unused_ -= it->first;
      kept_on(device) -= it->first;
      it = free_.erase(it);
    }
  }
  for (void* q : drop) (void)device_free(q);   // waits for the work that may still use it
  return !drop.empty();
}

bool MemPool::look(Clock::time_point now) {
  if (now - looked_ >= std::chrono::milliseconds(kLookMs)) {
    const size_t kept = kept_on(device);
    int current = -1;
    size_t free_now = 0, total = 0;
    if (hipGetDevice(&current) != hipSuccess || current != device ||
        hipMemGetInfo(&free_now, &total) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
    limit_ = std::min(kMax, (free_now + kept) / 8);
    looked_ = now;
  }
  return true;
}

void MemPool::trim() {
  std::multimap<size_t, Block> old;
  {
    std::lock_guard<std::mutex> hold(mu_);
    old.swap(free_);
    kept_on(device) -= unused_;
    unused_ = 0;
    looked_ = {};
  }
  for (auto& e : old) (void)device_free(e.second.p);   // waits for the work that may still use it
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
