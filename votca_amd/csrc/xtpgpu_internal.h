// Internal runtime pieces of libxtpgpu: error state, device buffers, context.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <array>
#include <atomic>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <stdexcept>
#include <string>
#include <utility>
#include <vector>

#include "../../include/xtpgpu.h"

namespace xg {

struct Error : public std::runtime_error {
  int code;
  Error(int c, const std::string& m) : std::runtime_error(m), code(c) {}
};

#define XG_HIP(expr)                                                                      \
  do {                                                                                    \
    hipError_t e_ = (expr);                                                               \
    if (e_ != hipSuccess) {                                                               \
      throw ::xg::Error(e_ == hipErrorOutOfMemory ? XTPGPU_ERR_OOM : XTPGPU_ERR_HIP,     \
                        std::string("HIP error '") + hipGetErrorString(e_) + "' at " +   \
                            __FILE__ + ":" + std::to_string(__LINE__) + " (" #expr ")"); \
    }                                                                                     \
  } while (0)

#define XG_REQUIRE(cond, code, msg)                        \
  do {                                                     \
    if (!(cond)) throw ::xg::Error((code), std::string(msg)); \
  } while (0)

// Large blocks (kMinBlock and more) that DevBufs of one device have given up, at most kBound bytes of them,
// the oldest freed first. Mapping and clearing device memory costs 0.2-10 ms per GiB, the more the process has
// mapped, and giving it back about as much: an operator's set-up of 2.1 GB (40 x 280 x 1280) takes 2.06 ms where it
// finds blocks that another of its size left, 2.4 where it does not, and 50 in a process with much memory mapped. A
// block enters once the device is idle, as hipFree would have waited, so whichever thread or stream
// takes it finds nothing still using it. drain() returns them: when a context lets go of its scratch or
// ends, and before an allocation of this library is refused (reclaim_current).
class BlockPool {
 public:
  static constexpr size_t kMinBlock = (size_t)16 << 20, kBound = (size_t)4 << 30;
  static BlockPool& of(int device) {
    static BlockPool* pools = new BlockPool[kDevices];  // not destroyed: buffers may outlive it at exit
    return pools[device];
  }
  BlockPool() { kept_.reserve(kBound / kMinBlock + 1); }  // give() runs in destructors: no allocation there
  static bool serves(int device) { return device >= 0 && device < kDevices; }
  // the smallest kept block of n to n + n / 8 bytes, or null
  void* take(size_t n, size_t& cap) {
    std::lock_guard<std::mutex> lk(mu_);
    size_t best = kept_.size();
    for (size_t i = 0; i < kept_.size(); ++i)
      if (kept_[i].cap >= n && kept_[i].cap <= n + n / 8 && (best == kept_.size() || kept_[i].cap < kept_[best].cap))
        best = i;
    if (best == kept_.size()) return nullptr;
    void* p = kept_[best].p;
    cap = kept_[best].cap;
    total_ -= cap;
    kept_.erase(kept_.begin() + best);
    return p;
  }
  // false: not taken in, the caller frees it
  bool give(int device, void* p, size_t cap) {
    if (cap > kBound) return false;
    int cur = device;
    if (hipGetDevice(&cur) != hipSuccess) return false;
    if (cur != device && hipSetDevice(device) != hipSuccess) return false;
    // hipFree waits for the device; hipDeviceSynchronize would, too, but it breaks off every stream capture of
    // the process, also another thread's thread-local one, beside which memory may be allocated and freed.
    // Allocating and freeing one byte takes 1.4 us on an idle device.
    void* mark = nullptr;
    const bool idle = hipMalloc(&mark, 1) == hipSuccess && hipFree(mark) == hipSuccess;
    if (!idle) (void)hipGetLastError();
    if (cur != device) (void)hipSetDevice(cur);
    if (!idle) return false;
    std::lock_guard<std::mutex> lk(mu_);
    while (!kept_.empty() && total_ + cap > kBound) free_oldest();
    kept_.push_back({p, cap});
    total_ += cap;
    return true;
  }
  void drain() {
    std::lock_guard<std::mutex> lk(mu_);
    while (!kept_.empty()) free_oldest();
  }

 private:
  static constexpr int kDevices = 64;
  struct Block {
    void* p;
    size_t cap;
  };
  void free_oldest() {
    (void)hipFree(kept_.front().p);
    total_ -= kept_.front().cap;
    kept_.erase(kept_.begin());
  }
  std::mutex mu_;
  std::vector<Block> kept_;
  size_t total_ = 0;
};

// Owning device allocation. The allocation checks free memory first, mirroring the
// reference's guard in CudaMatrix (xtp/src/libxtp/cudamatrix.cc:97-113).
struct DevBuf {
  void* p = nullptr;
  size_t bytes = 0;
  size_t cap = 0;   // bytes of the block, at least `bytes`
  int device = -1;  // of a block that the pool takes back
  DevBuf() = default;
  explicit DevBuf(size_t n) { alloc(n); }
  DevBuf(const DevBuf&) = delete;
  DevBuf& operator=(const DevBuf&) = delete;
  DevBuf(DevBuf&& o) noexcept { swap(o); }
  DevBuf& operator=(DevBuf&& o) noexcept {
    if (this != &o) { release(); swap(o); }
    return *this;
  }
  void swap(DevBuf& o) noexcept {
    std::swap(p, o.p); std::swap(bytes, o.bytes); std::swap(cap, o.cap); std::swap(device, o.device);
  }
  ~DevBuf() { release(); }
  void alloc(size_t n) {
    release();
    if (n == 0) return;
    // a query of the free memory costs 5-10 us, ten times a small allocation: below 1 MiB, where the
    // runtime mostly carves from a block that it holds, the allocation itself tells
    int dev = -1;
    if (n >= BlockPool::kMinBlock && hipGetDevice(&dev) == hipSuccess && BlockPool::serves(dev)) {
      p = BlockPool::of(dev).take(n, cap);
      if (p) {
        bytes = n;
        device = dev;
        return;
      }
    } else {
      dev = -1;
    }
    if (n >= ((size_t)1 << 20)) require_free(n);
    hipError_t rc = hipMalloc(&p, n);
    if (rc == hipErrorOutOfMemory) {
      (void)hipGetLastError();
      reclaim_current();
      require_free(n);
      rc = hipMalloc(&p, n);
    }
    if (rc != hipSuccess) p = nullptr;
    XG_HIP(rc);
    bytes = cap = n;
    device = dev;
  }
  static void drain_current() {
    int dev = -1;
    if (hipGetDevice(&dev) == hipSuccess && BlockPool::serves(dev)) BlockPool::of(dev).drain();
  }
  // what calls and destroyed objects have left for reuse on the current device goes back to it
  static void reclaim_current();
  // throws when the device has not got n bytes, what is kept given back
  static void require_free(size_t n) {
    size_t fr = 0, tot = 0;
    if (hipMemGetInfo(&fr, &tot) != hipSuccess || n <= fr) return;
    reclaim_current();
    if (hipMemGetInfo(&fr, &tot) == hipSuccess && n > fr)
      throw Error(XTPGPU_ERR_OOM, "device allocation of " + std::to_string(n) +
                                      " bytes exceeds free device memory (" + std::to_string(fr) + ")");
  }
  void ensure(size_t n) {
    if (n > bytes) alloc(n);
  }
  void release() {
    if (p && !(device >= 0 && BlockPool::of(device).give(device, p, cap))) (void)hipFree(p);
    p = nullptr;
    bytes = cap = 0;
    device = -1;
  }
  template <typename T> T* as() const { return reinterpret_cast<T*>(p); }
};

// Scratch that a context keeps between calls and that one call at a time uses.
struct KeptBuf {
  static constexpr size_t kKeepBytes = (size_t)256 << 20;
  DevBuf buf;
  std::atomic<bool> busy{false};
  void release() {
    if (busy.exchange(true)) return;  // in use by a call on another thread
    buf.release();
    busy.store(false);
  }
};

// The kept scratch of the living contexts, by device.
class KeptList {
 public:
  static KeptList& get() {
    static KeptList* list = new KeptList;  // not destroyed: contexts may outlive it at exit
    return *list;
  }
  void add(int device, KeptBuf* k) {
    std::lock_guard<std::mutex> lk(mu_);
    all_.push_back({device, k});
  }
  void remove(KeptBuf* k) {
    std::lock_guard<std::mutex> lk(mu_);
    for (size_t i = 0; i < all_.size(); ++i)
      if (all_[i].second == k) {
        all_.erase(all_.begin() + i);
        return;
      }
  }
  void release(int device) {
    std::lock_guard<std::mutex> lk(mu_);
    for (auto& e : all_)
      if (e.first == device) e.second->release();
  }

 private:
  std::mutex mu_;
  std::vector<std::pair<int, KeptBuf*>> all_;
};

inline void DevBuf::reclaim_current() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) return;
  KeptList::get().release(dev);
  drain_current();
}

// f() of another library that allocates for itself: once more with what is kept given back when it reports
// `no_memory` (before it has touched its operands)
template <class S, class F>
S with_reclaim(S no_memory, F f) {
  S s = f();
  if (s == no_memory) {
    DevBuf::reclaim_current();
    s = f();
  }
  return s;
}

// A call's scratch, for work on the context's stream only: the kept buffer, which the next call's work follows in
// the stream; or one of its own, for a call that finds the kept one in use (another thread) or needs more than
// is kept.
class Scratch {
 public:
  explicit Scratch(KeptBuf& k) : kept_(k.busy.exchange(true) ? nullptr : &k) {}
  ~Scratch() {
    if (kept_) kept_->busy.store(false);
  }
  Scratch(const Scratch&) = delete;
  Scratch& operator=(const Scratch&) = delete;
  unsigned char* get(size_t bytes) {
    DevBuf& b = kept_ && bytes <= KeptBuf::kKeepBytes ? kept_->buf : own_;
    b.ensure(bytes);
    return b.as<unsigned char>();
  }

 private:
  KeptBuf* kept_;
  DevBuf own_;
};

}  // namespace xg

namespace xg {
// Named kernel timers: HIP events recorded on the context's stream around tagged
// launches, with the algorithmic FLOPs / bytes of each launch.
struct KTimer {
  struct Rec { hipEvent_t a, b; double flops, bytes; };
  std::vector<Rec> pending;
  double ms = 0.0, flops = 0.0, bytes = 0.0;
  long launches = 0;
};
}  // namespace xg

struct xtpgpu_ctx_s {
  int device = 0;
  hipStream_t stream = nullptr;
  // grow-only scratch buffers, reused across calls on this context (ws[1]: the eps builds' scaled
  // transition copies, at most the scale budget)
  xg::DevBuf ws[3];
  // the adjoint's intermediates; partial sums of the self-energy and of operator diagonals; what eps builds
  // stage; vectors of products on host arrays
  xg::KeptBuf adjoint_ws, sum_ws, eps_ws, host_ws;
  std::array<xg::KeptBuf*, 4> kept() { return {&adjoint_ws, &sum_ws, &eps_ws, &host_ws}; }
  ~xtpgpu_ctx_s() {
    for (xg::KeptBuf* k : kept()) xg::KeptList::get().remove(k);
  }
  int cus = 256;  // compute units of the device
  // pinned memory for small host transfers (HostIo), allocated at the first one. It is used by the call
  // that set io_busy, until its end; a call that finds it set does without
  static constexpr size_t kPinBytes = (size_t)1 << 20;  // each way
  std::atomic<bool> io_busy{false};
  unsigned char* pin = nullptr;
  unsigned char* pin_dev = nullptr;  // as the device sees it
  bool profiling = false;
  void* blas = nullptr;  // rocblas_handle for the rocSOLVER calls, bound to `stream`
  std::vector<std::pair<std::string, xg::KTimer>> timers;
  std::vector<hipEvent_t> event_pool;
  xg::KTimer& timer(const std::string& n) {
    for (auto& t : timers)
      if (t.first == n) return t.second;
    timers.emplace_back(n, xg::KTimer());
    return timers.back().second;
  }
  hipEvent_t event() {
    if (!event_pool.empty()) {
      hipEvent_t e = event_pool.back();
      event_pool.pop_back();
      return e;
    }
    hipEvent_t e;
    XG_HIP(hipEventCreate(&e));
    return e;
  }
  // fold finished event pairs into the totals (call after the stream is synchronized)
  void collect() {
    for (auto& t : timers) {
      for (auto& r : t.second.pending) {
        float ms = 0.f;
        XG_HIP(hipEventElapsedTime(&ms, r.a, r.b));
        t.second.ms += ms;
        t.second.flops += r.flops;
        t.second.bytes += r.bytes;
        t.second.launches += 1;
        event_pool.push_back(r.a);
        event_pool.push_back(r.b);
      }
      t.second.pending.clear();
    }
  }
};

namespace xg {
// RAII scope that brackets the launches issued inside it with an event pair.
struct ProfScope {
  xtpgpu_ctx_s* c = nullptr;
  KTimer* t = nullptr;
  hipEvent_t a = nullptr;
  double flops, bytes;
  ProfScope(xtpgpu_ctx_s* ctx, const char* name, double f, double by) : flops(f), bytes(by) {
    if (ctx && ctx->profiling && name) {
      c = ctx;
      t = &ctx->timer(name);
      a = ctx->event();
      XG_HIP(hipEventRecord(a, ctx->stream));
    }
  }
  ~ProfScope() {
    if (c) {
      hipEvent_t b = c->event();
      if (hipEventRecord(b, c->stream) == hipSuccess) t->pending.push_back({a, b, flops, bytes});
    }
  }
};
}  // namespace xg

struct xtpgpu_mmn_s {
  xtpgpu_ctx ctx = nullptr;
  int device = 0;  // the context's, which may end first (an interpreter's exit finalises objects in any order)
  int64_t mmin = 0, mmax = 0, nmin = 0, nmax = 0, mtotal = 0, ntotal = 0, aux = 0;
  // Device layout, aux-major: element (m, n, P) at data[P*mtotal*ntotal + m*ntotal + n].
  xg::DevBuf data;
  uint64_t version = 0;  // bumped whenever the tensor changes
  double* d() const { return data.as<double>(); }
  size_t pstride() const { return (size_t)mtotal * (size_t)ntotal; }
};
