// From-all pull of a small graph in one launch per level, the functor's
// filter included.
//
// Where the sources' state stays in the caches, gathering it per edge is cheaper
// than propagation blocking's two passes over per-edge messages, whose pieces
// also leave most of the chip idle on a small graph. Targets are listed once per
// graph by in-degree: a lane takes a row of up to 8 edges, eight lanes one of
// up to 128, a wavefront one of up to 2048, a workgroup a longer one, so that
// every row is summed in one place and the rank update can follow at once. The
// update writes the other of two source-state arrays (the messages of the same
// level still read the first), which then change places.
// Latency bounds it: a list entry, row offsets, columns and messages are a
// chain of four loads.
// Which graphs: the gathers gain where they stay in the caches, that is with
// few sources, with few edges, or with sources that concentrate on part of the
// lines (hubs with neighbouring ids) or follow the rows (a grid); a sample of
// the in-edges tells the last (rows_cover). Measured per PageRank iteration, us,
// propagation blocking -> whole rows:
//   few sources      uniform random, 64 K of them: 2.1 M edges 22 -> 13, 8.4 M 50 -> 43;
//                    128 K: 2.1 M 20 -> 17, 4.2 M 25 -> 22, 8.4 M 41 -> 40; but
//                    256 K: 2.1 M 20 -> 20, 4.2 M 24 -> 29
//   few edges        random, 1 M sources: 1 M edges 25 -> 17, 2.1 M 26 -> 24, 3.1 M 25 -> 30
//   concentrated     R-MAT 19 to 22, 7 to 8.3 M edges: 58 -> 38, 71 -> 46, 83 -> 57, 114 -> 76;
//                    grid 1400 x 1400 78 -> 27
//   spread           random, 8.4 M edges, 512 K / 1 M / 2 M sources: 39 -> 52, 42 -> 74, 51 -> 104;
//                    R-MAT 19 to 22 with shuffled ids 36 -> 47, 44 -> 57, 56 -> 72, 81 -> 110;
//                    preferential attachment, 1 M sources 46 -> 59
// The sample covers 0.08 (grids) to 0.30 of the lines on the concentrated graphs
// and 0.45 to 0.63 on the spread ones, hence the line at 3/8.
// Not where one row is long, since one workgroup walks it, 0.6 us per 1024
// edges, while propagation blocking splits it. Stars: 16 K leaves 35 -> 14, 32 K
// 34 -> 23, 65 K 35 -> 43, 262 K 36 -> 161; a row of 1/128 of all edges ends with
// the others.
#pragma once
#include "expand_pull.h"
#include "pb.h"

namespace gsw {

constexpr int ROWS_CLASSES = 4;
constexpr int ROWS_LANE = 8, ROWS_GROUP = 128, ROWS_WAVE = 2048;  // longest row of a class
constexpr int64_t ROWS_MAX_EDGES = 8 << 20;
constexpr int64_t ROWS_FEW_SOURCES = 128 << 10, ROWS_FEW_EDGES = 2 << 20;
constexpr int64_t ROWS_LONGEST = 32 << 10;
constexpr double ROWS_COVER = 0.375;
constexpr int ROWS_LINE = 128;  // bytes of a cache line

__device__ __forceinline__ int rows_class(int64_t deg) {
  return deg <= ROWS_LANE ? 0 : deg <= ROWS_GROUP ? 1 : deg <= ROWS_WAVE ? 2 : 3;
}

// pass 0: class sizes into cnt[0..4), the longest row above ROWS_WAVE into
// cnt[4]; pass 1: rows into list, class k from cnt[k] on (the offsets, moved
// along)
__global__ void __launch_bounds__(BLOCK)
    k_rows_list(const int64_t *__restrict__ rows, int64_t n, int32_t *list,
                unsigned long long *cnt) {
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> LOG_WAVE;
  for (int64_t base = wave << 6; base < n; base += nwaves << 6) {
    const int64_t v = base + lane;
    const int64_t deg = v < n ? rows[v + 1] - rows[v] : -1;
    const int c = v < n ? rows_class(deg) : -1;
    if (!list && deg > ROWS_WAVE) atomicMax(cnt + ROWS_CLASSES, (unsigned long long)deg);
#pragma unroll
    for (int k = 0; k < ROWS_CLASSES; ++k) {
      const uint64_t m = ballot(c == k);
      if (!m) continue;
      unsigned long long at = 0;
      if (lane == 0) at = atomicAdd(cnt + k, (unsigned long long)__popcll(m));
      at = __shfl(at, 0, 64);
      if (list && c == k) list[at + rank_below(m)] = (int32_t)v;
    }
  }
}

// class sizes and the longest row, once per graph
inline void rows_count(rowbins_t &rb, const int64_t *rows, int64_t n) {
  if (rb.longest >= 0) return;
  unsigned long long *cnt = nullptr, h[ROWS_CLASSES + 1];
  H_ERR(hipMalloc((void **)&cnt, sizeof(h)));
  try {
    fill_async<unsigned long long>(cnt, 0ull, ROWS_CLASSES + 1);
    hipLaunchKernelGGL(k_rows_list, dim3(grid_for((n + 63) / 64 * 64)), dim3(BLOCK), 0, stream(),
                       rows, n, (int32_t *)nullptr, cnt);
    H_ERR(hipGetLastError());
    H_ERR(hipMemcpyAsync(h, cnt, sizeof(h), hipMemcpyDeviceToHost, stream()));
    sync();
  } catch (...) {
    (void)hipFree(cnt);
    throw;
  }
  H_ERR(hipFree(cnt));
  int64_t at = 0;
  for (int k = 0; k < ROWS_CLASSES; ++k) {
    rb.off[k] = at;
    rb.cnt[k] = (int64_t)h[k];
    at += rb.cnt[k];
  }
  GSW_REQUIRE(at == n, E_INTERNAL_CHECK, "row classes miss rows");
  rb.longest = (int64_t)h[ROWS_CLASSES];
}

inline void rows_ensure(rowbins_t &rb, const int64_t *rows, int64_t n) {
  if (rb.list) return;
  rows_count(rb, rows, n);
  unsigned long long *cnt = nullptr, off[ROWS_CLASSES];
  for (int k = 0; k < ROWS_CLASSES; ++k) off[k] = (unsigned long long)rb.off[k];
  int32_t *list = nullptr;
  H_ERR(hipMalloc((void **)&cnt, sizeof(off)));
  try {
    H_ERR(hipMalloc((void **)&list, sizeof(int32_t) * (n + 1)));
    H_ERR(hipMemcpyAsync(cnt, off, sizeof(off), hipMemcpyHostToDevice, stream()));
    hipLaunchKernelGGL(k_rows_list, dim3(grid_for((n + 63) / 64 * 64)), dim3(BLOCK), 0, stream(),
                       rows, n, list, cnt);
    H_ERR(hipGetLastError());
    sync();
  } catch (...) {
    (void)hipFree(cnt);
    (void)hipFree(list);
    throw;
  }
  H_ERR(hipFree(cnt));
  rb.list = list;
}

// A sample of the in-edges, as many as the source state has lines, one wavefront
// per window of 64 consecutive ones: *count += lines touched. `bits`: one per
// line, zero before. Sources spread evenly touch 1 - 1/e = 0.63 of the lines.
__global__ void __launch_bounds__(BLOCK)
    k_rows_cover(const int32_t *__restrict__ cols, int64_t m, int64_t windows, int per_line,
                 uint32_t *bits, unsigned long long *count) {
  const int64_t w = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  if (w >= windows) return;
  const int64_t at = windows > 1 ? w * (m - WAVE) / (windows - 1) : 0;
  const int line = cols[at + lane_id()] / per_line;
  const uint32_t bit = 1u << (line & 31);
  const uint64_t first = ballot(!(atomicOr(bits + (line >> 5), bit) & bit));
  if (lane_id() == 0 && first) atomicAdd(count, (unsigned long long)__popcll(first));
}

// The share of the source state's lines that the sample touches, once per
// graph (m >= WAVE; `src_bytes`: of one source's state).
inline double rows_cover(rowbins_t &rb, const int32_t *cols, int64_t n, int64_t m,
                         int src_bytes) {
  if (rb.cover >= 0) return rb.cover;
  const int per = MAX(1, ROWS_LINE / src_bytes);
  const int64_t lines = (n + per - 1) / per, words = (lines + 31) / 32 + 1;
  const int64_t windows = MAX((int64_t)1, MIN(lines, m) / WAVE);
  unsigned long long *tmp = nullptr, h = 0;  // the count, then the bits
  H_ERR(hipMalloc((void **)&tmp, sizeof(*tmp) + sizeof(uint32_t) * words));
  try {
    uint32_t *bits = (uint32_t *)(tmp + 1);
    fill_async<uint32_t>((uint32_t *)tmp, 0u, words + 2);
    hipLaunchKernelGGL(k_rows_cover, dim3((unsigned)((windows * WAVE + BLOCK - 1) / BLOCK)),
                       dim3(BLOCK), 0, stream(), cols, m, windows, per, bits, tmp);
    H_ERR(hipGetLastError());
    H_ERR(hipMemcpyAsync(&h, tmp, sizeof(h), hipMemcpyDeviceToHost, stream()));
    sync();
  } catch (...) {
    (void)hipFree(tmp);
    throw;
  }
  H_ERR(hipFree(tmp));
  return rb.cover = (double)h / (double)lines;
}

// Whether whole rows are the faster pull of a graph (the reasons and both
// sides' times are above). GSW_ROWS_EDGES: by that number of edges alone, for
// sweeps.
inline bool rows_wanted(rowbins_t &rb, const int64_t *rows, const int32_t *cols, int64_t n,
                        int64_t m, int src_bytes) {
  if (const char *e = std::getenv("GSW_ROWS_EDGES")) return m <= std::atoll(e);
  if (m > ROWS_MAX_EDGES) return false;
  rows_count(rb, rows, n);
  if (rb.longest > MAX(ROWS_LONGEST, m / 128)) return false;
  if (n <= ROWS_FEW_SOURCES || m <= ROWS_FEW_EDGES) return true;
  return rows_cover(rb, cols, n, m, src_bytes) < ROWS_COVER;
}

// workgroups of each class
inline int rows_blocks(const rowbins_t &rb, int k) {
  const int per[ROWS_CLASSES] = {BLOCK, BLOCK / 8, BLOCK / WAVE, 1};
  return (int)((rb.cnt[k] + per[k] - 1) / per[k]);
}

// the messages of in-edges [s, e) of one row, lane `i` of `w`
template <class Bd>
__device__ __forceinline__ typename Bd::WA rows_sum(Bd &body, int64_t s, int64_t e, int i,
                                                    int w) {
  typename Bd::WA acc{};
  for (int64_t j = s + i; j < e; j += 4 * w) {
    int u[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) u[r] = j + r * w < e ? body.cols()[j + r * w] : -1;
    typename Bd::WA m[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) m[r] = body.msg(u[r] >= 0 ? u[r] : u[0], 0);
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (u[r] >= 0) body.f.comp(&acc, m[r], body.g);
  }
  return acc;
}

// `out`: the functor whose filter writes the other source-state array.
template <class Bd, class F>
__global__ void __launch_bounds__(BLOCK)
    k_pull_rows(Bd body, F out, rowbins_t rb, int4 first_block) {
  const unsigned long long t0 = wall_clock64();
  using WA = typename Bd::WA;
  __shared__ WA s_part[BLOCK / WAVE];
  const int b = blockIdx.x, t = threadIdx.x;
  // longest rows first: first_block holds the first workgroup of classes 2, 1, 0
  const int k = b < first_block.x ? 3 : b < first_block.y ? 2 : b < first_block.z ? 1 : 0;
  const int bk = b - (k == 3 ? 0 : k == 2 ? first_block.x : k == 1 ? first_block.y : first_block.z);
  const int w = k == 0 ? 1 : k == 1 ? 8 : k == 2 ? WAVE : BLOCK;  // threads per row
  const int64_t i = (int64_t)bk * (BLOCK / w) + t / w;
  const bool ok = i < rb.cnt[k];
  int v = 0;
  int64_t s = 0, e = 0;
  if (ok) {
    v = rb.list[rb.off[k] + i];
    s = body.rows()[v];
    e = body.rows()[v + 1];
  }
  WA acc = rows_sum(body, s, e, t % w, w);
  for (int o = MIN(w, WAVE) >> 1; o > 0; o >>= 1) {
    const WA x = shfl_xor_any(acc, o);
    body.f.comp(&acc, x, body.g);
  }
  if (k == 3) {  // uniform over the workgroup
    if (lane_id() == 0) s_part[t >> LOG_WAVE] = acc;
    __syncthreads();
    acc = s_part[0];
    for (int j = 1; j < BLOCK / WAVE; ++j) body.f.comp(&acc, s_part[j], body.g);
  }
  if (ok && t % w == 0) {
    *out.ra_of(v) = *body.f.ra_of(v);
    (void)out.filter_acc(v, acc, body.g);
  }
  add_work(body.as.dg_work, t0, ok && t % w == 0 ? (unsigned long long)(e - s) : 0ull, 0ull);
}

}  // namespace gsw
