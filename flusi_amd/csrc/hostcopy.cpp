// Copies of large fields between the device and the caller's (pageable) FP64
// host arrays.
//
// A plain hipMemcpy to a fresh pageable array ran at 10 GB/s (3.2 GB: 306 ms):
// one thread moves the data out of the runtime's staging buffers and takes the
// array's page faults, and a single-precision field crossed the bus as FP64.
// Here several threads each keep two chunks in flight through pinned slots of
// their own and move (FP32 fields: widen or narrow) them to or from the
// caller's array: page faults and conversion run on all of them beside the
// transfers, and FP32 fields cross the bus in FP32.  FP64, fresh array, 4 MB
// chunks, eight threads: 3.2 GB 306 -> 69 ms, 403 MB 39 -> 9.1 ms, 101 MB 9.7
// -> 2.6 ms (four threads: 78, 10.4, 2.8 ms).
//
// Smaller copies stay plain (kStagedBytes): alone they gain, too (18.9 MB 1.8
// -> 0.8 ms), but beside a program whose own thread pool still spins on every
// core after its last parallel loop, a thread of this copy can wait a time
// slice of a few milliseconds for a core (three 19 MB copies of a host
// program between conversions of its own: 3.1 -> 6.4 ms with threads).  Slots
// driven by the calling thread alone were not measured.
//
// The pinned slots cost 4 ms (64 MB) when they are made and first touched, once
// while contexts of a device live.  Copies out into fresh arrays regain that at
// once (into arrays touched before they do not: 115 MB of an FP32 field, whose
// first copy took 2 ms more than a plain one).  Copies in do only from some size
// on (kMakeIn): a smaller one that finds no slots is left to the plain copy
// once, for a program that sets one state and steps on (50 MB of FP64: in
// 1.8 ms plain, 5.1 ms with the slots to be made, 1.4 ms with slots there).
#include "hostcopy.h"
#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <sched.h>
#include <system_error>
#include <thread>
#include <type_traits>
#include <vector>

namespace flusi {

namespace {

constexpr int kMaxThreads = 8;
constexpr size_t kStagedBytes = 48u << 20;  // transfers from which the threads pay
constexpr size_t kMakeIn[2] = {96u << 20, 320u << 20};  // FP32, FP64 transfers in that regain the slots' making
// bytes of a slot: half the slots' cost for the smaller transfers, which run as
// fast with 2 MB (50 MB of FP64: out 1.6 / 1.9 ms, in 1.42 / 1.36); larger ones
// do not (403 MB: 35 / 21 ms)
size_t slot_bytes(size_t transfer) { return transfer < (96u << 20) ? 2u << 20 : 4u << 20; }

// makes a device current for this thread while alive
struct DeviceScope {
  int old = -1;
  hipError_t status;
  explicit DeviceScope(int d) {
    if ((status = hipGetDevice(&old)) == hipSuccess && old != d) status = hipSetDevice(d);
    else old = -1;
  }
  ~DeviceScope() { if (old >= 0) (void)hipSetDevice(old); }
};

// pinned slots and their events, two per thread
struct Ring {
  const size_t slot;
  char* mem = nullptr;
  hipEvent_t ev[2 * kMaxThreads] = {};
  explicit Ring(size_t bytes) : slot(bytes) {}
  ~Ring() {
    for (hipEvent_t e : ev) if (e) (void)hipEventDestroy(e);
    if (mem) (void)hipHostFree(mem);
  }
  hipError_t init() {
    for (hipEvent_t& e : ev)
      if (hipError_t r = hipEventCreateWithFlags(&e, hipEventDisableTiming)) return r;
    return hipHostMalloc((void**)&mem, slot * 2 * kMaxThreads, hipHostMallocDefault);
  }
};

int cpus() {
  cpu_set_t set;
  const int n = sched_getaffinity(0, sizeof(set), &set) == 0 ? CPU_COUNT(&set) : 1;
  return std::max(1, n);
}

}  // namespace

// Keeps one idle ring; concurrent copies beyond it bring their own.
class HostCopyPool {
 public:
  explicit HostCopyPool(int d) : device(d) {}
  const int device;
  // A ring for `transfer` bytes.  make: one is made where there is none or only
  // one of smaller slots; else a smaller one serves, and where there is none
  // the first call gets none.  Null also: no pinned memory or events to be had.
  std::unique_ptr<Ring> take(size_t transfer, bool make) {
    const size_t slot = slot_bytes(transfer);
    std::unique_ptr<Ring> r;
    {
      std::lock_guard<std::mutex> g(mu_);
      r = std::move(idle_);
      if (!r && !make && !declined_) {
        declined_ = true;
        return r;
      }
    }
    if (r && (!make || r->slot >= slot)) return r;
    r.reset();  // (its memory first)
    r.reset(new Ring(slot));
    if (r->init() != hipSuccess) {
      (void)hipGetLastError();  // not the next call's error
      r.reset();
    }
    return r;
  }
  void give(std::unique_ptr<Ring> r) {
    std::lock_guard<std::mutex> g(mu_);
    if (!idle_ || idle_->slot < r->slot) std::swap(idle_, r);
  }

 private:
  std::mutex mu_;
  std::unique_ptr<Ring> idle_;
  bool declined_ = false;  // a copy has been left to the plain copy for want of a ring
};

std::shared_ptr<HostCopyPool> host_copy_pool(int d) {
  static std::mutex mu;
  static std::map<int, std::weak_ptr<HostCopyPool>> pools;
  std::lock_guard<std::mutex> g(mu);
  std::shared_ptr<HostCopyPool> p = pools[d].lock();
  if (!p) pools[d] = p = std::make_shared<HostCopyPool>(d);
  return p;
}

namespace {

template <typename D, typename S> void convert(D* dst, const S* src, size_t n) {
  if constexpr (std::is_same<D, S>::value) std::memcpy(dst, src, n * sizeof(D));
  else for (size_t i = 0; i < n; ++i) dst[i] = (D)src[i];
}

// Runs work(worker) on up to `threads` threads, this one among them; a thread
// that cannot be started leaves its chunks to the others.
template <typename F> void run_workers(int threads, F&& work) {
  std::vector<std::thread> t;
  t.reserve(kMaxThreads);
  for (int w = 1; w < threads; ++w) {
    try {
      t.emplace_back(work, w);
    } catch (const std::system_error&) {
      break;
    }
  }
  work(0);
  for (std::thread& x : t) x.join();
}

// out: device -> host, else host -> device
template <typename T, bool OUT>
bool staged(HostCopyPool& pool, T* dev, double* host, long n, hipStream_t s, hipError_t& result) {
  const DeviceScope scope(pool.device);  // the ring's events are the stream's device's
  const size_t bytes = (size_t)n * sizeof(T);
  std::unique_ptr<Ring> ring = pool.take(bytes, OUT || bytes >= kMakeIn[sizeof(T) == 8]);
  if (!ring) return false;
  const long per = (long)(ring->slot / sizeof(T)), chunks = (n + per - 1) / per;
  const int threads = (int)std::min<long>({(long)kMaxThreads, (long)cpus(), (chunks + 1) / 2});
  std::atomic<long> next{0};
  std::atomic<int> err{(int)hipSuccess};
  auto check = [&](hipError_t e) {
    int ok = (int)hipSuccess;
    if (e != hipSuccess) err.compare_exchange_strong(ok, (int)e);
    return e == hipSuccess;
  };
  auto work = [&](int w) {
    const DeviceScope on(pool.device);
    if (!check(on.status)) return;
    long c[2] = {-1, -1};  // the chunk in each slot
    auto len = [&](long k) { return (size_t)std::min(per, n - k * per); };
    auto slot = [&](int i) { return reinterpret_cast<T*>(ring->mem + (size_t)(2 * w + i) * ring->slot); };
    auto fetch = [&](int i) {  // the next chunk into slot i
      const long k = next.fetch_add(1);
      if (k >= chunks || err.load() != (int)hipSuccess) return false;
      c[i] = k;
      if (!OUT) convert(slot(i), host + k * per, len(k));
      const hipError_t e = OUT ? hipMemcpyAsync(slot(i), dev + k * per, len(k) * sizeof(T), hipMemcpyDeviceToHost, s)
                               : hipMemcpyAsync(dev + k * per, slot(i), len(k) * sizeof(T), hipMemcpyHostToDevice, s);
      return check(e) && check(hipEventRecord(ring->ev[2 * w + i], s));
    };
    for (int i = 0; i < 2; ++i)
      if (!fetch(i)) break;
    for (int i = 0; c[i] >= 0; i ^= 1) {
      const long k = c[i];
      c[i] = -1;
      if (!check(hipEventSynchronize(ring->ev[2 * w + i]))) return;
      if (OUT) convert(host + k * per, slot(i), len(k));
      (void)fetch(i);
    }
  };
  run_workers(threads, work);
  // (also after an error: no transfer may outlive the ring)
  const hipError_t e = hipStreamSynchronize(s);
  if (e == hipSuccess && err.load() == (int)hipSuccess) pool.give(std::move(ring));
  result = err.load() != (int)hipSuccess ? (hipError_t)err.load() : e;
  return true;
}

}  // namespace

// Host memory that the runtime knows needs no staging: the plain copy goes
// straight to pinned memory (FP64, 256^3 velocity: out 8.5 ms, staged 9.3; state
// in 7.1 / 9.0) and leaves managed or device memory to the runtime.  FP32
// fields still cross the bus in half the bytes (out 7.9 / 5.1, in 7.2 / 4.9).
bool host_copy_pays(const void* host, long n, size_t elem) {
  if ((size_t)n * elem < kStagedBytes) return false;
  hipPointerAttribute_t a{};
  if (hipPointerGetAttributes(&a, host) != hipSuccess) {
    (void)hipGetLastError();  // (one answer for ordinary memory)
    return true;
  }
  return a.type == hipMemoryTypeUnregistered || (a.type == hipMemoryTypeHost && elem == sizeof(float));
}

template <typename T>
bool host_copy_out(HostCopyPool& pool, const T* dev, double* host, long n, hipStream_t s, hipError_t& result) {
  return staged<T, true>(pool, const_cast<T*>(dev), host, n, s, result);
}
template <typename T>
bool host_copy_in(HostCopyPool& pool, const double* host, T* dev, long n, hipStream_t s, hipError_t& result) {
  return staged<T, false>(pool, dev, const_cast<double*>(host), n, s, result);
}

template bool host_copy_out<float>(HostCopyPool&, const float*, double*, long, hipStream_t, hipError_t&);
template bool host_copy_out<double>(HostCopyPool&, const double*, double*, long, hipStream_t, hipError_t&);
template bool host_copy_in<float>(HostCopyPool&, const double*, float*, long, hipStream_t, hipError_t&);
template bool host_copy_in<double>(HostCopyPool&, const double*, double*, long, hipStream_t, hipError_t&);

}  // namespace flusi
