// Shared internals of libsucem_hip: error state, device buffers, context.
#pragma once
#include <hip/hip_runtime.h>

#include <chrono>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "sucem_hip.h"

namespace sucem {

// Error carrying a C-ABI status code.
struct Error : std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

void set_last_error(const std::string& msg);

#define SUCEM_HIP(call)                                                           \
  do {                                                                            \
    hipError_t e_ = (call);                                                       \
    if (e_ != hipSuccess) {                                                       \
      throw ::sucem::Error(e_ == hipErrorOutOfMemory ? SUCEM_ERR_OOM : SUCEM_ERR_HIP, \
                           std::string(#call) + ": " + hipGetErrorString(e_) +     \
                               " (" __FILE__ ":" + std::to_string(__LINE__) + ")"); \
    }                                                                             \
  } while (0)

#define SUCEM_CHECK(cond, code, msg)                    \
  do {                                                  \
    if (!(cond)) throw ::sucem::Error((code), (msg));   \
  } while (0)

// Device memory that a context's finished buffers leave for its next ones.  Building a mesh,
// a space and a system takes some 250 buffers, most of them for one step; allocated and
// freed one by one they cost 15 of the 25 ms of an order-2 set-up of 32,400 cells (hipFree
// also waits for the whole device).
//
// A block that is put back may still be in use by work queued on its context's stream, so it
// is only handed out to that context (whose stream orders the new use behind the old one).
// Whoever frees memory that other streams may use has the device waited for first, as hipFree
// does: the destroy entry points (DeviceWait) and members replaced while their owner lives
// (DBuf::release_synced).  All pools of a device together keep at most kMax bytes unused, and
// at most an eighth of the memory that would be free without them: allocations outside the
// library (torch's) cannot make a pool give way.  Blocks go back to the device beyond that (those
// first that nobody has asked for in a second: a program that went on to other meshes would
// otherwise find the pools full of sizes that it no longer needs), when the context's workspace
// is released, when free memory is asked for, when an allocation of the library fails (all
// pools give way), and with the context (buffers that outlive it free directly).
class MemPool {
 public:
  static constexpr size_t kMax = size_t(4) << 30;
  ~MemPool();
  // a block of at least `bytes` (its size in `got`), or throws SUCEM_ERR_OOM
  void* take(size_t bytes, size_t& got);
  void put(void* p, size_t size);
  void trim();    // everything unused back to the device
  void close();   // trim, and keep nothing from now on
  size_t unused();
  int device = -1;   // of its context

 private:
  using Clock = std::chrono::steady_clock;
  struct Block {
    void* p;
    Clock::time_point since;
  };
  bool keep(void* p, size_t size, Clock::time_point now);
  bool drop_idle(Clock::time_point now);   // blocks unused for kIdleMs; whether there were any
  bool look(Clock::time_point now);        // limit_ up to date, if the device says so
  static constexpr int kIdleMs = 1000;
  std::mutex mu_;
  std::multimap<size_t, Block> free_;
  Clock::time_point oldest_{};             // no block has been unused for longer
  size_t unused_ = 0;
  // The device's free memory is looked at again after kLookMs: a look takes 5 to 11 us, and
  // one for every 64 MB that came back made up 3 % of a far-field transform.
  static constexpr int kLookMs = 50;
  size_t limit_ = 0;
  Clock::time_point looked_{};
  bool closed_ = false;
};
// The pool of the context that this thread's current entry point runs on (Context::use).
std::shared_ptr<MemPool>& current_pool();
std::shared_ptr<MemPool> new_pool();
// every pool of a device gives its unused blocks back
void trim_pools(int device);
// hipMalloc; when it fails, once more after every pool has given its unused blocks back
void* device_alloc(size_t bytes);
// hipFree (which waits for all work on the device); a refusal leaves no error behind for the
// thread's next launch to report
bool device_free(void* p);

// While it lives, this thread's allocations and frees are neither refused because of another
// stream's capture nor end it (they belong to no graph).
class BesideCaptures {
 public:
  BesideCaptures() {
    if (hipThreadExchangeStreamCaptureMode(&mode_) != hipSuccess) {
      (void)hipGetLastError();
      changed_ = false;
    }
  }
  ~BesideCaptures() {
    if (changed_) (void)hipThreadExchangeStreamCaptureMode(&mode_);
  }

 private:
  hipStreamCaptureMode mode_ = hipStreamCaptureModeRelaxed;
  bool changed_ = true;
};

// Waits until the device's queued work is done, before buffers that any stream may use go back
// to their pools.  Through hipFree of a small block (1.2 us on an idle device, some 100 us behind
// a stream that has not been waited for, so the owner's stream is waited for first): a
// hipDeviceSynchronize ends every stream capture of the process, that of another thread's
// batched sweep among them.  Should that be refused, the buffers that this thread releases
// while the object lives go to the device instead, which orders them itself.
class DeviceWait {
 public:
  explicit DeviceWait(hipStream_t owners);
  ~DeviceWait() { bypass_pools() = before_; }
  static bool& bypass_pools();   // of this thread

 private:
  bool before_;
};

// Owning device allocation.
template <typename T>
struct DBuf {
  T* p = nullptr;
  size_t n = 0;
  size_t size = 0;                  // of the block
  std::shared_ptr<MemPool> pool;    // where the block goes back to (null: to the device)
  DBuf() = default;
  explicit DBuf(size_t count) { alloc(count); }
  DBuf(const DBuf&) = delete;
  DBuf& operator=(const DBuf&) = delete;
  DBuf(DBuf&& o) noexcept : p(o.p), n(o.n), size(o.size), pool(std::move(o.pool)) {
    o.p = nullptr;
    o.n = o.size = 0;
  }
  DBuf& operator=(DBuf&& o) noexcept {
    if (this != &o) {
      release();
      p = o.p; n = o.n; size = o.size; pool = std::move(o.pool);
      o.p = nullptr;
      o.n = o.size = 0;
    }
    return *this;
  }
  ~DBuf() { release(); }
  void alloc(size_t count, bool pooled = true) {
    release();
    if (count) {
      std::shared_ptr<MemPool> from = pooled ? current_pool() : nullptr;
      size = count * sizeof(T);
      p = (T*)(from ? from->take(size, size) : device_alloc(size));
      pool = std::move(from);
    }
    n = count;
  }
  void release() {
    if (p) {
      if (pool && !DeviceWait::bypass_pools()) pool->put(p, size);
      else (void)device_free(p);
    }
    p = nullptr;
    n = size = 0;
    pool.reset();
  }
  // release of memory that work on another context's stream may still use: to the device,
  // which waits for it
  void release_synced() {
    pool.reset();
    release();
  }
  size_t bytes() const { return n * sizeof(T); }
};

// Device workspace of a context: numbered slots that keep their allocation from call to
// call and grow when a call needs more, so repeated solves on one context allocate (and
// free, which synchronises the device) nothing after the first.  A slot is used by one
// routine at a time: the Krylov solver takes slots [0, 32) and 84, the eigen solver [32, 48) (it
// calls the Krylov solver, so their ranges differ), the batched solver [48, 80), the point entry
// points [80, 84), operator products of several vectors 85.  Calls on one context run one at a time (one host thread per context).
struct Workspace {
  std::vector<DBuf<unsigned char>> slot;
  // device memory of at least `bytes` bytes in slot k (nullptr for 0 bytes); the contents
  // are whatever the slot's last user left
  void* get(int k, size_t bytes) {
    if (bytes == 0) return nullptr;
    if ((size_t)k >= slot.size()) slot.resize(k + 1);
    if (slot[k].n < bytes) {
      slot[k].release();
      // 1/8 headroom for a slightly larger next call; not from the pool, which is for
      // buffers that come and go
      slot[k].alloc(bytes + (bytes >> 3), false);
    }
    return slot[k].p;
  }
  size_t bytes() const {
    size_t t = 0;
    for (const auto& b : slot) t += b.n;
    return t;
  }
  void release() { slot.clear(); }
};

struct Context {
  int device = 0;
  hipStream_t stream = nullptr;
  bool own_stream = false;
  int num_cus = 256;
  // pinned host staging for scalar readbacks
  double* pinned = nullptr;
  size_t pinned_n = 0;
  Workspace ws;
  std::shared_ptr<MemPool> pool = new_pool();
  // library-owned stream (non-blocking, default priority) for work captured in hipGraphs:
  // the caller's stream may be the null stream, which cannot be captured
  hipStream_t aux_stream = nullptr;
  hipStream_t graph_stream() {
    if (!aux_stream) SUCEM_HIP(hipStreamCreateWithFlags(&aux_stream, hipStreamNonBlocking));
    return aux_stream;
  }
  void sync() { SUCEM_HIP(hipStreamSynchronize(stream)); }
  void use() {
    SUCEM_HIP(hipSetDevice(device));
    current_pool() = pool;
  }
  double* host_scratch(size_t n);
  // One value from a kernel to the host without a copy: next_mail numbers the message and
  // gives the kernel its address in pinned memory (a value and a sequence number), wait_mail
  // waits until that message has arrived and returns its value.
  double* mail_h = nullptr;   // host and device view of the two words
  double* mail_d = nullptr;
  unsigned long long mail_seq = 0;
  double* next_mail(unsigned long long& seq);
  double wait_mail();
};

// typed view of workspace slot k holding `count` elements
template <typename T>
inline T* ws_take(Context* c, int k, int64_t count) {
  return (T*)c->ws.get(k, count > 0 ? sizeof(T) * (size_t)count : 0);
}

// `count` elements for one call: workspace slot k up to 32 MB, beyond that an allocation
// that is given back with the call (the workspace is not to hold an occasional large call)
template <typename T>
struct Scratch {
  DBuf<T> own;
  T* p = nullptr;
  Scratch(Context* c, int k, int64_t count) {
    if (count > 0 && sizeof(T) * (size_t)count <= (size_t(32) << 20)) {
      p = ws_take<T>(c, k, count);
    } else {
      own.alloc(count > 0 ? (size_t)count : 0);
      p = own.p;
    }
  }
};

template <typename T>
inline void h2d(Context* c, T* d, const T* h, size_t n) {
  if (n) SUCEM_HIP(hipMemcpyAsync(d, h, n * sizeof(T), hipMemcpyHostToDevice, c->stream));
}
template <typename T>
inline void d2h(Context* c, T* h, const T* d, size_t n) {
  if (n) SUCEM_HIP(hipMemcpyAsync(h, d, n * sizeof(T), hipMemcpyDeviceToHost, c->stream));
}

inline unsigned grid_for(int64_t n, int block, int64_t cap = 1 << 20) {
  int64_t g = (n + block - 1) / block;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}

#define SUCEM_LAUNCH(kernel, grid, block, shmem, stream, ...)                          \
  do {                                                                                 \
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(block), shmem, stream, __VA_ARGS__);  \
    SUCEM_HIP(hipGetLastError());                                                      \
  } while (0)

}  // namespace sucem

// Opaque handle definitions (C-ABI types).
struct sucem_ctx {
  sucem::Context c;
};
