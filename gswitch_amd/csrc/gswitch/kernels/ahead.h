// Fused levels run ahead of the host.
//
// A fused level (push over the unsorted queue, next queue by de-duplicated
// appends) leaves the host nothing to decide but whether to go on, so waiting
// for its queue length only adds a round trip to every level. The executor
// therefore launches up to AHEAD levels in a row, one launch each: the
// ordinary fused WM push, which reads its queue length on the device, logs it
// with the clock and finds nothing to do once the frontier has drained or has
// outgrown the grid that the batch was launched with. The host waits once per
// batch. Queue lengths rotate through three slots (a level reads one, appends
// to the next and clears the one that its predecessor read), the queues and
// the de-duplication bitmaps through two.
// Measured: BFS on a 1500 x 1377 grid, 52 levels of up to 220 K vertices,
// 1673 -> 1233 us; SSSP on 1000 x 1023, 70 levels, 2787 -> 1840 us.
#pragma once
#include "../data_structures/active_set.h"
#include "../utils/runtime.h"
#include "expand_push.h"

namespace gsw {

constexpr int AHEAD = 8;  // levels per batch
constexpr int AHEAD_SLOTS = 3;

// Device words of a run of fused levels (the host reads them all).
struct ahead_t {
  long long clock[AHEAD];  // device clock when the batch's levels began
  int32_t sizes[AHEAD];    // their queue lengths
  int32_t q[AHEAD_SLOTS];  // rotating queue lengths
  int32_t pad;
};
static_assert(sizeof(ahead_t) % 8 == 0, "reported as 64-bit words");
constexpr int AHEAD_WORDS = sizeof(ahead_t) / 8;

// Input length nq into slot `in`, the others zero; both de-duplication bitmaps
// clean (n_bits words each; 0: left alone).
__global__ void __launch_bounds__(BLOCK)
    k_ahead_begin(ahead_t *a, int in, int nq, uint64_t *b0, uint64_t *b1, int64_t n_bits) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  for (int64_t i = t; i < n_bits; i += (int64_t)gridDim.x * blockDim.x) {
    b0[i] = 0;
    b1[i] = 0;
  }
  if (t < AHEAD_SLOTS) a->q[t] = t == in ? nq : 0;
}

// Level j of a batch, input length in slot `in`; `reach`: the most frontier
// vertices that this grid is meant for.
template <class B>
__global__ void __launch_bounds__(BLOCK)
    k_push_wm_ahead(B body, int vpw, ahead_t *a, int j, int in, int reach) {
  const int N = a->q[in];
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    a->sizes[j] = N;
    a->clock[j] = (long long)wall_clock64();
    a->q[(in + 2) % AHEAD_SLOTS] = 0;
  }
  if (N == 0 || N > reach) return;  // the whole grid
  push_wm_range(body, vpw, N);
}

// End of a batch: the words, the clock and the overflow flag to the host.
__global__ void __launch_bounds__(64)
    k_ahead_end(const ahead_t *a, const int32_t *ctrl, long long *host, long long *mark,
                long long seq) {
  const int t = threadIdx.x;
  if (t < AHEAD_WORDS) host[t] = ((const long long *)a)[t];
  if (t == AHEAD_WORDS) host[t] = (long long)wall_clock64();
  if (t == AHEAD_WORDS + 1) host[t] = ctrl[CTRL_OVERFLOW];
  __threadfence_system();
  __syncthreads();
  if (t == 0) publish(mark, seq);
}

}  // namespace gsw
