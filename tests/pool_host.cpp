// The device memory pools (csrc/mempool.cpp) over a counted stand-in for the device: one named
// check per run, exit code 0 when it holds.  Built and run by tests/test_pool_host.py.
#include <cstdlib>
#include <map>
#include <set>
#include <thread>

#include "mempool.cpp"

namespace {

struct Device {
  size_t capacity = size_t(288) << 30, used = 0, next = 4096;
  std::map<size_t, size_t> blocks;   // address -> bytes
  int mallocs = 0, frees = 0;
  bool refuse = false;   // as under another stream's global capture
  hipStreamCaptureMode mode = hipStreamCaptureModeGlobal;   // of the thread
  hipError_t last = hipSuccess;
} dev;

hipError_t fail(hipError_t e) { return dev.last = e; }

}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) {
  if (dev.refuse) return fail(hipErrorStreamCaptureUnsupported);
  if (dev.used + bytes > dev.capacity) return fail(hipErrorOutOfMemory);
  ++dev.mallocs;
  *p = (void*)dev.next;
  dev.blocks[dev.next] = bytes;
  dev.next += bytes + 4096;
  dev.used += bytes;
  return hipSuccess;
}
hipError_t hipFree(void* p) {
  if (dev.refuse) return fail(hipErrorStreamCaptureUnsupported);
  auto it = dev.blocks.find((size_t)p);
  if (it == dev.blocks.end()) std::abort();   // freed twice, or never allocated
  ++dev.frees;
  dev.used -= it->second;
  dev.blocks.erase(it);
  return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
  if (dev.refuse) return fail(hipErrorStreamCaptureImplicit);
  *s = hipStreamCaptureStatusNone;
  return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError(void) {
  const hipError_t e = dev.last;
  dev.last = hipSuccess;
  return e;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = dev.capacity - dev.used;
  *t = dev.capacity;
  return hipSuccess;
}
hipError_t hipGetDevice(int* d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipThreadExchangeStreamCaptureMode(hipStreamCaptureMode* m) {
  std::swap(*m, dev.mode);
  return hipSuccess;
}
// ends every capture of the process: nothing here may call it
hipError_t hipDeviceSynchronize(void) { std::abort(); }
const char* hipGetErrorString(hipError_t) { return "stand-in error"; }
}

using namespace sucem;

namespace {

constexpr size_t MB = size_t(1) << 20, GB = size_t(1) << 30;

struct Fixture {
  std::shared_ptr<MemPool> pool = new_pool();
  Fixture() {
    pool->device = 0;
    current_pool() = pool;
  }
};

#define CHECK(cond)                                               \
  do {                                                            \
    if (!(cond)) {                                                \
      std::printf("line %d: %s is false\n", __LINE__, #cond);     \
      return 1;                                                   \
    }                                                             \
  } while (0)

// blocks come back from the pool, and only to a request of about their size
int reuse() {
  Fixture f;
  void* p;
  {
    DBuf<char> a(10 * MB);
    p = a.p;
  }
  CHECK(f.pool->unused() >= 10 * MB && dev.frees == 0);
  {
    DBuf<char> a(10 * MB);
    CHECK(a.p == p && dev.mallocs == 1 && f.pool->unused() == 0);
    DBuf<char> b(8 * MB);
    CHECK(dev.mallocs == 2);
  }
  DBuf<char> c(5 * MB);   // neither 10 nor 8 MB for 5
  CHECK(dev.mallocs == 3);
  return 0;
}

// at most kMax bytes stay in a pool, beyond that blocks go back to the device
int cap() {
  Fixture f;
  {
    std::vector<DBuf<char>> a;
    for (int i = 0; i < 12; ++i) a.emplace_back(512 * MB);
    CHECK(dev.used >= 6 * GB);
  }
  CHECK(f.pool->unused() <= MemPool::kMax && f.pool->unused() > MemPool::kMax - 640 * MB);
  CHECK(dev.used == f.pool->unused());
  {
    DBuf<char> big(MemPool::kMax + 1);
  }
  CHECK(dev.used == f.pool->unused() && f.pool->unused() <= MemPool::kMax);
  return 0;
}

// trim and close give everything back; a closed pool keeps nothing
int trim() {
  Fixture f;
  {
    DBuf<char> a(MB), b(3 * MB);
  }
  CHECK(f.pool->unused() > 0);
  f.pool->trim();
  CHECK(f.pool->unused() == 0 && dev.used == 0);
  DBuf<char> late(2 * MB);
  f.pool->close();
  late.release();
  CHECK(dev.used == 0 && f.pool->unused() == 0);
  return 0;
}

// a failed allocation empties every pool of the process and is tried again
int full_device() {
  Fixture f;
  auto other = new_pool();
  other->device = 0;
  {
    DBuf<char> a(2 * GB);
    current_pool() = other;
    DBuf<char> b(GB);
  }
  CHECK(f.pool->unused() + other->unused() >= 3 * GB);
  dev.capacity = 6 * GB;
  current_pool() = f.pool;
  DBuf<char> big(5 * GB);
  CHECK(f.pool->unused() == 0 && other->unused() == 0 && dev.last == hipSuccess);
  bool thrown = false;
  try {
    DBuf<char> more(5 * GB);
  } catch (const Error& e) {
    thrown = e.code == SUCEM_ERR_OOM;
  }
  CHECK(thrown);
  return 0;
}

// what a buffer takes from the device: at most an eighth more than its size (512 bytes for the
// smallest), the size itself beyond what a pool can keep, also when a kept block is handed out
int rounding() {
  Fixture f;
  for (size_t n : {size_t(1), size_t(511), size_t(4096), size_t(4097), size_t(8191), size_t(8193),
                   size_t(1000003), 16 * MB + 1, 3 * GB + 12345, MemPool::kMax}) {
    const size_t used = dev.used;
    DBuf<char> a(n);
    const size_t took = dev.used - used;
    CHECK(took >= n && took - n <= std::max(n / 8, size_t(511)));
    a.release();
    f.pool->trim();
  }
  {
    const size_t used = dev.used;
    DBuf<char> a(MemPool::kMax + 1);
    CHECK(dev.used - used == MemPool::kMax + 1);
  }
  for (size_t n = 100; n < 64 * MB; n = n * 5 / 4 + 1) {   // blocks of every class, kept
    DBuf<char> a(n);
  }
  for (size_t n = 4096; n < 40 * MB; n = n * 9 / 8 + 7) {
    DBuf<char> a(n);
    CHECK(a.size >= n && a.size - n <= n / 8);
  }
  f.pool->trim();
  // a request for what is left gets it although its rounded size does not fit
  dev.capacity = dev.used + 9 * MB + 4;
  DBuf<char> exact(9 * MB + 4);
  CHECK(exact.p && exact.size == 9 * MB + 4 && dev.last == hipSuccess);
  return 0;
}

// the pools of a device keep kMax bytes together, and little of a device that is nearly full
int shared_cap() {
  Fixture f;
  std::vector<std::shared_ptr<MemPool>> pools;
  size_t kept = 0;
  for (int i = 0; i < 3; ++i) {
    pools.push_back(new_pool());
    pools.back()->device = 0;
    current_pool() = pools.back();
    std::vector<DBuf<char>> a;
    for (int j = 0; j < 5; ++j) a.emplace_back(512 * MB);
    a.clear();
    kept += pools.back()->unused();
  }
  CHECK(kept <= MemPool::kMax && kept > MemPool::kMax - 512 * MB && dev.used == kept);
  trim_pools(0);
  CHECK(dev.used == 0);
  for (auto& q : pools) CHECK(q->unused() == 0);
  // 8 GB free: an eighth of them may be kept, whatever is asked for
  dev.capacity = 8 * GB;
  const auto look = std::chrono::milliseconds(60);   // its free memory is looked at again
  for (int round = 0; round < 3; ++round) {
    std::vector<DBuf<char>> a;
    for (int j = 0; j < 40; ++j) a.emplace_back(96 * MB);
    std::this_thread::sleep_for(look);
    a.clear();
    CHECK(dev.used <= GB && dev.used >= GB / 4);
  }
  std::this_thread::sleep_for(look);
  DBuf<char>(96 * MB).release();   // looked at with nothing in use
  {
    std::vector<DBuf<char>> a;
    for (int j = 0; j < 40; ++j) a.emplace_back(96 * MB);
  }
  CHECK(dev.used <= GB && dev.used >= 3 * GB / 4);
  // memory that others take lowers it
  dev.capacity = dev.used + 2 * GB;
  std::this_thread::sleep_for(look);
  for (int round = 0; round < 3; ++round) {
    std::vector<DBuf<char>> a;
    for (int j = 0; j < 20; ++j) a.emplace_back(96 * MB);
  }
  CHECK(dev.used <= GB / 2);
  pools.clear();
  current_pool().reset();
  f.pool.reset();
  CHECK(dev.used == 0 && dev.mode == hipStreamCaptureModeGlobal);
  return 0;
}

// a full pool makes room by giving back what nobody has asked for in a second, its own and
// other pools' blocks, and nothing younger
int idle() {
  Fixture f;
  auto other = new_pool();
  other->device = 0;
  auto fill = [&](const std::shared_ptr<MemPool>& p, int n, size_t size) {
    current_pool() = p;
    std::vector<DBuf<char>> a;
    for (int i = 0; i < n; ++i) a.emplace_back(size);
  };
  fill(f.pool, 4, 512 * MB);
  fill(other, 4, 512 * MB);
  CHECK(dev.used == 4 * GB && f.pool->unused() + other->unused() == 4 * GB);
  fill(f.pool, 1, 96 * MB);
  CHECK(dev.used == 4 * GB);   // full, and nothing is old: the block went back
  std::this_thread::sleep_for(std::chrono::milliseconds(1100));
  fill(other, 1, 512 * MB);    // in use again: young
  fill(f.pool, 1, 96 * MB);
  CHECK(f.pool->unused() == 96 * MB && other->unused() == 512 * MB);
  CHECK(dev.used == 608 * MB);
  fill(f.pool, 20, 160 * MB);
  CHECK(dev.used <= 4 * GB && f.pool->unused() > 3 * GB && other->unused() == 512 * MB);
  return 0;
}

// blocks are pooled after a wait for the device; where the wait is refused they never reach a
// pool, and no error is left for the next launch
int wait() {
  Fixture f;
  DBuf<char> a(MB), b(MB), c(MB);
  {
    const int frees = dev.frees;
    const DeviceWait w(nullptr);
    CHECK(dev.frees == frees + 1);   // hipFree waits
    a.release();
  }
  CHECK(f.pool->unused() >= MB);
  const size_t idle = f.pool->unused();
  {
    dev.refuse = true;
    const DeviceWait w(nullptr);
    b.release();
  }
  CHECK(f.pool->unused() == idle && dev.last == hipSuccess);
  dev.refuse = false;
  {
    const DeviceWait w(nullptr);
  }
  {
    const int frees = dev.frees;
    c.release_synced();
    CHECK(dev.frees == frees + 1 && f.pool->unused() == idle && !c.p);
  }
  DBuf<char> d(2 * MB);
  d.release();   // the refusal is over
  CHECK(f.pool->unused() > idle);
  return 0;
}

}  // namespace

int main(int argc, char** argv) {
  const std::map<std::string, int (*)()> checks = {
      {"reuse", reuse}, {"cap", cap}, {"trim", trim}, {"full_device", full_device},
      {"wait", wait}, {"rounding", rounding},
      {"shared_cap", shared_cap}, {"idle", idle}};
  auto it = argc == 2 ? checks.find(argv[1]) : checks.end();
  if (it == checks.end()) return 2;
  return it->second();
}
