// CPU stand-in for <hip/hip_runtime.h>, used ONLY by the host-compiled test build of the
// kernels.  One std::thread per GPU thread, blocks run one after another, so the
// kernels' own index arithmetic, masking and LDS traffic run unchanged under the host
// AddressSanitizer.  Nothing in the shipped library includes this file.
#pragma once
#include <atomic>
#include <barrier>
#include <cassert>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <dlfcn.h>
#include <map>
#include <memory>
#include <mutex>
#include <sched.h>
#include <string>
#include <thread>
#include <vector>

#define __global__
#define __device__
#define __host__
#define __forceinline__ inline __attribute__((always_inline))
#define __launch_bounds__(...)
#define __shared__ static

struct dim3 {
  unsigned x, y, z;
  dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct EmuIdx { unsigned x = 0, y = 0, z = 0; };
inline thread_local EmuIdx threadIdx, blockIdx, blockDim, gridDim;

typedef int hipError_t;
typedef void* hipStream_t;
enum { hipSuccess = 0, hipErrorOutOfMemory = 2 };
inline hipError_t hipGetLastError() { return hipSuccess; }
// Launches run at once and in order, so streams and events order nothing here; what the calls would order is written down:
// per stream the launches given to it, per event the stream and its count when it was recorded, per pair of streams how far
// the first waits for the second.
typedef void* hipEvent_t;
enum { hipEventDisableTiming = 2 };
struct EmuOrder {
  std::mutex lock;
  uintptr_t handles = 0;
  long long allowed = -1;                // events that can still be made (-1: any number)
  std::map<hipStream_t, long long> given;
  std::map<hipEvent_t, std::pair<hipStream_t, long long>> events;
  std::map<std::pair<hipStream_t, hipStream_t>, long long> waited;
};
inline EmuOrder emu_order;
inline void emu_note_launch(hipStream_t s) {
  std::lock_guard<std::mutex> l(emu_order.lock);
  emu_order.given[s]++;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
  std::lock_guard<std::mutex> l(emu_order.lock);
  if (emu_order.allowed == 0) return hipErrorOutOfMemory;
  if (emu_order.allowed > 0) emu_order.allowed--;
  *e = reinterpret_cast<hipEvent_t>(++emu_order.handles);
  return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
  std::lock_guard<std::mutex> l(emu_order.lock);
  emu_order.events[e] = {s, emu_order.given[s]};
  return hipSuccess;
}
inline hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
  std::lock_guard<std::mutex> l(emu_order.lock);
  auto it = emu_order.events.find(e);
  if (it != emu_order.events.end()) emu_order.waited[{s, it->second.first}] = it->second.second;
  return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t e) {
  std::lock_guard<std::mutex> l(emu_order.lock);
  emu_order.events.erase(e);
  return hipSuccess;
}
extern "C" inline __attribute__((used)) void amoe_emu_allow_events(long long n) {
  std::lock_guard<std::mutex> l(emu_order.lock);
  emu_order.allowed = n;
}
// launches given to `other`, and how many of them stream s does not wait for
extern "C" inline __attribute__((used)) long long amoe_emu_launches(hipStream_t other) {
  std::lock_guard<std::mutex> l(emu_order.lock);
  return emu_order.given[other];
}
extern "C" inline __attribute__((used)) long long amoe_emu_not_waited_for(hipStream_t s, hipStream_t other) {
  std::lock_guard<std::mutex> l(emu_order.lock);
  return emu_order.given[other] - emu_order.waited[{s, other}];
}
inline const char* hipGetErrorString(hipError_t) { return "emu"; }
enum hipDeviceAttribute_t { hipDeviceAttributeMultiprocessorCount = 0 };
inline hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
// a "device" array is ordinary host memory here, and its address is the symbol's own
#define __align__(n) __attribute__((aligned(n)))
#define HIP_SYMBOL(x) (&(x))
template <class T> inline hipError_t hipGetSymbolAddress(void** p, T* sym) { *p = (void*)sym; return hipSuccess; }
// A 3-CU device: the persistent kernels then run few workgroups with several work items each.  AMOE_EMU_CUS: another one,
// for the launches that depend on how many there are (asked for once, by the first launch of a process).
inline hipError_t hipDeviceGetAttribute(int* v, hipDeviceAttribute_t, int) {
  const char* cus = getenv("AMOE_EMU_CUS");
  *v = cus ? atoi(cus) : 3;
  return hipSuccess;
}
// symbol of the kernel that was launched last
inline std::string emu_last_kernel;
extern "C" inline __attribute__((used)) const char* amoe_emu_last_kernel() { return emu_last_kernel.c_str(); }

// Barrier for heavily oversubscribed threads (256 per workgroup on a few cores): waiters give up the core instead of
// sleeping on a futex, which costs two system calls and a wake-up per thread and barrier.
struct EmuBarrier {
  explicit EmuBarrier(int n_) : n(n_) {}
  void arrive_and_wait() {
    const unsigned g = gen.load(std::memory_order_acquire);
    if (count.fetch_add(1, std::memory_order_acq_rel) + 1 == n) {
      count.store(0, std::memory_order_relaxed);
      gen.fetch_add(1, std::memory_order_release);
    } else {
      while (gen.load(std::memory_order_acquire) == g) sched_yield();
    }
  }
  const int n;
  std::atomic<int> count{0};
  std::atomic<unsigned> gen{0};
};

struct EmuWave {
  EmuBarrier bar{64};
  alignas(64) unsigned char slot[64][64];
  const void* ptr[64];
};
struct EmuBlock {
  EmuBarrier* bar;
};
inline thread_local EmuWave* emu_wave = nullptr;
inline thread_local EmuBlock* emu_block = nullptr;

inline void __syncthreads() { emu_block->bar->arrive_and_wait(); }

template <class T> inline T atomicAdd(T* p, T v) { return __atomic_fetch_add(p, v, __ATOMIC_RELAXED); }
inline float atomicAdd(float* p, float v) {
  std::atomic_ref<float> r(*p);
  float old = r.load();
  while (!r.compare_exchange_weak(old, old + v)) {}
  return old;
}
inline void __threadfence() { __atomic_thread_fence(__ATOMIC_SEQ_CST); }
template <class T> inline T atomicOr(T* p, T v) { return __atomic_fetch_or(p, v, __ATOMIC_RELAXED); }
template <class T> inline T atomicMax(T* p, T v) {
  T old = __atomic_load_n(p, __ATOMIC_RELAXED);
  while (old < v && !__atomic_compare_exchange_n(p, &old, v, true, __ATOMIC_RELAXED, __ATOMIC_RELAXED)) {}
  return old;
}

template <class K, class... A>
inline void emu_launch(K kernel, dim3 grid, dim3 block, A... args) {
  const unsigned nthreads = block.x;
  assert(nthreads % 64 == 0 && block.y == 1 && block.z == 1);
  Dl_info symbol{};
  emu_last_kernel = dladdr(reinterpret_cast<const void*>(kernel), &symbol) && symbol.dli_sname ? symbol.dli_sname : "";
  for (unsigned bz = 0; bz < grid.z; bz++)
  for (unsigned by = 0; by < grid.y; by++)
  for (unsigned bx = 0; bx < grid.x; bx++) {
    EmuBarrier bar((int)nthreads);
    EmuBlock blk{&bar};
    std::unique_ptr<EmuWave[]> waves(new EmuWave[nthreads / 64]);
    std::vector<std::thread> th;
    th.reserve(nthreads);
    for (unsigned t = 0; t < nthreads; t++) {
      th.emplace_back([&, t]() {
        threadIdx.x = t;
        blockIdx.x = bx; blockIdx.y = by; blockIdx.z = bz;
        blockDim.x = nthreads; blockDim.y = blockDim.z = 1;
        gridDim.x = grid.x; gridDim.y = grid.y; gridDim.z = grid.z;
        emu_wave = &waves[t / 64];
        emu_block = &blk;
        kernel(args...);
      });
    }
    for (auto& x : th) x.join();
  }
}
#define hipLaunchKernelGGL(kernel, grid, block, shmem, stream, ...) \
  (emu_note_launch(stream), emu_launch(kernel, grid, block, __VA_ARGS__))
