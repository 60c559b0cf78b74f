// Process-wide runtime pieces: the engine's HIP stream, fill kernels and
// small launch helpers. All engine work is ordered on one stream per device;
// host reads of device scalars go through pinned memory + one stream sync.
#pragma once
#include "common.h"

namespace gsw {

inline hipStream_t &stream_slot() {
  static thread_local hipStream_t s = nullptr;
  return s;
}

// The stream every engine launch uses (created on first use, default
// priority, blocking w.r.t. the null stream so plain hipMemcpy orders with it).
inline hipStream_t stream() {
  hipStream_t &s = stream_slot();
  if (!s) H_ERR(hipStreamCreate(&s));
  return s;
}

template <typename T>
__global__ void k_fill(T *__restrict__ p, T val, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n; i += stride) p[i] = val;
}

inline int grid_for(int64_t work, int block = BLOCK, int max_grid = MAX_GRID) {
  int64_t g = (work + block - 1) / block;
  if (g < 1) g = 1;
  if (g > max_grid) g = max_grid;
  return (int)g;
}

// Device-side fill (a kernel, not hipMemsetAsync, so it can live in a
// captured graph).
template <typename T> inline void fill_async(T *p, T val, int64_t n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill<T>, dim3(grid_for(n)), dim3(BLOCK), 0, stream(),
                     p, val, n);
  H_ERR(hipGetLastError());
}

template <typename T> inline void set_one_async(T *p, T val) {
  hipLaunchKernelGGL(k_fill<T>, dim3(1), dim3(64), 0, stream(), p, val,
                     (int64_t)1);
  H_ERR(hipGetLastError());
}

inline void sync() { H_ERR(hipStreamSynchronize(stream())); }

// A kernel's small results reach the host through pinned memory: the kernel
// stores them, then (publish) a mark that the host polls for. Against a copy
// and a stream synchronisation this takes the copy's launch and the wake-up
// out of every level (52 fused levels of BFS on a 1500 x 1377 grid: 41 -> 28 us
// each, the profiling events gone as well). Called by one thread, after the
// workgroup's other threads' stores to host memory are fenced and joined.
template <typename T> __device__ __forceinline__ void publish(T *mark, T seq) {
  __threadfence_system();
  __hip_atomic_store(mark, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Host side: until *mark == seq. A stream that failed, or ended without the
// mark, is an error and not an endless wait.
template <typename T> inline void await_mark(const T *mark, T seq, hipStream_t st) {
  for (int64_t spin = 1; __atomic_load_n(mark, __ATOMIC_ACQUIRE) != seq; ++spin) {
    __builtin_ia32_pause();
    if (spin % 65536 == 0) {
      const hipError_t e = hipStreamQuery(st);
      if (e == hipErrorNotReady) continue;
      H_ERR(e);
      GSW_REQUIRE(__atomic_load_n(mark, __ATOMIC_ACQUIRE) == seq, E_HIP,
                  "a kernel's result did not arrive");
    }
  }
}

// words[0..n) of device memory to pinned host memory, then the mark
template <typename T>
__global__ void __launch_bounds__(64)
    k_report(const T *__restrict__ a, int na, const T *__restrict__ b, int nb, T *host,
             T *mark, T seq) {
  for (int i = threadIdx.x; i < na + nb; i += blockDim.x)
    host[i] = i < na ? a[i] : b[i - na];
  __threadfence_system();
  __syncthreads();
  if (threadIdx.x == 0) publish(mark, seq);
}

// Pinned host staging for small device->host reads.
struct pinned_t {
  void *p = nullptr;
  size_t bytes = 0;
  void *get(size_t b) {
    if (b > bytes) {
      if (p) hipHostFree(p);
      H_ERR(hipHostMalloc(&p, b));
      bytes = b;
    }
    return p;
  }
  ~pinned_t() {
    if (p) hipHostFree(p);
  }
};

}  // namespace gsw
