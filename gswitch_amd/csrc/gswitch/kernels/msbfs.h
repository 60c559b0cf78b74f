// 64-source bitmask BFS (multi-source BFS with one uint64 per vertex).
//
// No counterpart kernel in the reference (application/mbfs.cu runs the same
// single-source BFS three times); this is the batched form of its BFS: bit s
// of visit[v] is set once v is reachable from source s, bit s of front[v]
// once v was first reached from s at the previous level. A level is either
//  pull: every vertex with unvisited source bits ORs its neighbours' front
//        masks (stopping once all its open bits are covered);
//  push: every vertex with a non-empty front ORs it into its neighbours'
//        next masks (64-bit atomicOr), then a sweep keeps the new bits.
// Rows of more than MS_WIDE edges are cut into chunks of MS_CHUNK edges,
// listed once per graph, and a level spreads the chunks over the grid, one
// wavefront each: on R-MAT the hubs have the smallest ids, so the wavefront
// of word 0 used to walk 64 hub rows alone (R-MAT 20, edge factor 16: the
// first pull level took 2.6-9.7 ms, now 0.25 ms).
// Per level the kernels also count, per source, how many vertices were newly
// reached (a 64x64 bit transpose and one popcount per wavefront), from which
// the host builds a per-source sum of levels -- a checksum of all 64 BFS
// trees.
#pragma once
#include "../utils/runtime.h"
#include "../utils/wave.h"

namespace gsw {

constexpr int MS_WIDE = 64;     // degree above which a row is cut into chunks
constexpr int MS_CHUNK = 1024;  // edges per chunk of a wide row

struct ms_counters_t {
  unsigned long long newly;         // vertices with new bits this level
  unsigned long long newly_deg;     // their degree sum
  unsigned long long per_src[64];   // newly reached vertices per source
  unsigned long long pad[14];       // one slot = five 128-byte lines
};
// Workgroups add their counts into one of MS_SLOTS partial copies (slot
// blockIdx.x % MS_SLOTS); k_msbfs_finish sums and clears them. Atomics that
// every workgroup of the grid sends to the same lines serialise on MI355X.
constexpr int MS_SLOTS = 64;
static_assert(sizeof(ms_counters_t) == 640, "slot size");

// Per-source counts of the 64 lanes' `bits`; lane s accumulates source s.
// A 64x64 bit transpose (six exchange steps) puts source s's bits of all
// lanes into lane s: about 90 instructions per word with any new bit and
// none without, where 64 ballots cost 1000 for every word (R-MAT 20: a sweep
// that finds nothing 20.2 -> 4.3 us).
__device__ __forceinline__ void ms_count_sources(uint64_t bits,
                                                 unsigned long long &cnt) {
  if (!ballot(bits != 0ull)) return;
  const int lane = lane_id();
  constexpr uint64_t M[6] = {0x00000000FFFFFFFFull, 0x0000FFFF0000FFFFull,
                             0x00FF00FF00FF00FFull, 0x0F0F0F0F0F0F0F0Full,
                             0x3333333333333333ull, 0x5555555555555555ull};
#pragma unroll
  for (int k = 0; k < 6; ++k) {
    const int j = 32 >> k;
    const uint64_t p = __shfl_xor(bits, j, 64);
    bits = (lane & j) ? (((p >> j) & M[k]) | (bits & ~M[k]))
                      : ((bits & M[k]) | ((p & M[k]) << j));
  }
  cnt += __popcll(bits);
}

// Workgroup reduction of the counts, then one set of atomics into the
// workgroup's slot. Every thread of the workgroup calls it.
__device__ __forceinline__ void ms_flush(ms_counters_t *c,
                                         unsigned long long newly,
                                         unsigned long long ndeg,
                                         unsigned long long cnt) {
  constexpr int NW = BLOCK / WAVE;
  __shared__ unsigned long long s_src[NW][WAVE];
  __shared__ unsigned long long s_tot[NW][2];
  const int w = threadIdx.x >> LOG_WAVE, lane = lane_id();
  newly = wave_sum_any(newly);
  ndeg = wave_sum_any(ndeg);
  s_src[w][lane] = cnt;
  if (lane == 0) {
    s_tot[w][0] = newly;
    s_tot[w][1] = ndeg;
  }
  __syncthreads();
  if (w == 0) {
    ms_counters_t *slot = c + (blockIdx.x & (MS_SLOTS - 1));
    unsigned long long t = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += s_src[i][lane];
    if (t) atomicAdd(&slot->per_src[lane], t);
    if (lane < 2) {
      unsigned long long x = 0;
#pragma unroll
      for (int i = 0; i < NW; ++i) x += s_tot[i][lane];
      if (x) atomicAdd(lane == 0 ? &slot->newly : &slot->newly_deg, x);
    }
  }
}

// ---- wide rows -------------------------------------------------------------
// The rows of more than MS_WIDE edges of one CSR: their vertices (any order),
// one (vertex index, chunk) entry per MS_CHUNK edges, and one mask per vertex
// that the pull's chunks combine into (zero between levels). cap_v and cap_e
// bound both lists from the edge count, so building them needs no host read.
struct ms_wide_t {
  int32_t *v = nullptr;
  int2 *ent = nullptr;
  unsigned long long *acc = nullptr;
  unsigned long long *cnt = nullptr;  // [0] vertices, [1] entries
  int64_t cap_v = 0, cap_e = 0;
};
inline int64_t ms_wide_cap_v(int64_t n, int64_t m) {
  return MIN(n, m / (MS_WIDE + 1)) + 1;
}
inline int64_t ms_wide_cap_e(int64_t n, int64_t m) {
  return ms_wide_cap_v(n, m) + m / MS_CHUNK;
}

__global__ void __launch_bounds__(BLOCK)
    k_msbfs_wide(const int64_t *__restrict__ rows, int64_t n, ms_wide_t wd) {
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> LOG_WAVE;
  for (int64_t base = wave << 6; base < n; base += nwaves << 6) {
    const int64_t v = base + lane;
    const int64_t deg = v < n ? rows[v + 1] - rows[v] : 0;
    const bool wide = deg > MS_WIDE;
    const uint64_t m = ballot(wide);
    if (!m) continue;
    const int nc = wide ? (int)((deg + MS_CHUNK - 1) / MS_CHUNK) : 0;
    int tot;
    const int ex = wave_exclusive_scan(nc, tot);
    unsigned long long bv = 0, be = 0;
    if (lane == 0) {
      bv = atomicAdd(wd.cnt, (unsigned long long)__popcll(m));
      be = atomicAdd(wd.cnt + 1, (unsigned long long)tot);
    }
    bv = __shfl(bv, 0, 64);
    be = __shfl(be, 0, 64);
    if (wide) {
      const int64_t k = (int64_t)bv + rank_below(m);
      if (k < wd.cap_v) {
        wd.v[k] = (int32_t)v;
        wd.acc[k] = 0ull;
      }
      for (int c = 0; c < nc; ++c) {
        const int64_t e = (int64_t)be + ex + c;
        if (e < wd.cap_e) wd.ent[e] = make_int2((int)k, c);
      }
    }
  }
}

// The wide rows' part of a pull: one wavefront per chunk, 256 edges per step
// (four independent column loads, then four mask gathers per lane). A chunk
// stops once its vertex's open bits are covered, by itself or by the chunks
// that finished before it.
__global__ void __launch_bounds__(BLOCK)
    k_msbfs_pull_wide(const int64_t *__restrict__ rows, const int32_t *__restrict__ cols,
                      uint64_t all, const uint64_t *__restrict__ visit,
                      const uint64_t *__restrict__ front, ms_wide_t wd) {
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> LOG_WAVE;
  const int64_t ne = (int64_t)wd.cnt[1];
  for (int64_t i = wave; i < ne; i += nwaves) {
    const int2 e = wd.ent[i];
    const int v = wd.v[e.x];
    const uint64_t open = all & ~visit[v];
    if (!open) continue;
    const int64_t s = rows[v] + (int64_t)e.y * MS_CHUNK;
    const int64_t end = MIN(rows[v + 1], s + MS_CHUNK);
    // (lane 0's value for all: the loop below is uniform over the wavefront)
    const uint64_t had = __shfl(
        __hip_atomic_load(wd.acc + e.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), 0, 64);
    uint64_t got = had;
    for (int64_t j0 = s; j0 < end && (got & open) != open; j0 += 4 * WAVE) {
      int u[4];
      uint64_t x = 0;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const int64_t j = j0 + k * WAVE + lane;
        u[k] = j < end ? cols[j] : -1;
      }
#pragma unroll
      for (int k = 0; k < 4; ++k) x |= u[k] >= 0 ? front[u[k]] : 0ull;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) x |= __shfl_xor(x, o, 64);
      got |= x;
    }
    got &= open;
    if (lane == 0 && (got & ~had)) atomicOr(wd.acc + e.x, (unsigned long long)got);
  }
}

// Bottom-up level over the in-edges (rows/cols: the reverse CSR of a
// directed graph). Writes next[v] = newly reached bits for every v and
// counts the out-degrees (out_rows) of the newly reached vertices, the
// next level's push work. Wide rows (has_wide) take the masks that
// k_msbfs_pull_wide left in wd.acc and clear them; the others are walked by
// one lane each, four edges per step so that a lane's dependent chain of a
// column and a mask load is a quarter as long.
__global__ void __launch_bounds__(BLOCK)
    k_msbfs_pull(const int64_t *__restrict__ rows,
                 const int32_t *__restrict__ cols,
                 const int64_t *__restrict__ out_rows, int64_t n, uint64_t all,
                 uint64_t *__restrict__ visit,
                 const uint64_t *__restrict__ front,
                 uint64_t *__restrict__ next, ms_counters_t *c, bool has_wide,
                 ms_wide_t wd) {
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> LOG_WAVE;
  unsigned long long newly = 0, ndeg = 0, cnt = 0;
  for (int64_t base = wave << 6; base < n; base += nwaves << 6) {
    const int64_t v = base + lane;
    uint64_t vis = all, acc = 0;
    int64_t s = 0, e = 0;
    bool wide = false;
    if (v < n) {
      s = rows[v];
      e = rows[v + 1];
      // (not by visit[v]: the loop below writes a wide row's visit and next
      // while other wavefronts are still here)
      wide = (e - s) > MS_WIDE;
      if (!wide) vis = visit[v];
    }
    const uint64_t open = all & ~vis;
    if (open)
      for (int64_t j = s; j < e; j += 4) {
        int u[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) u[k] = j + k < e ? cols[j + k] : -1;
#pragma unroll
        for (int k = 0; k < 4; ++k) acc |= u[k] >= 0 ? front[u[k]] : 0ull;
        if ((acc & open) == open) break;
      }
    const uint64_t nw = acc & open;
    if (v < n && !wide) {
      next[v] = nw;
      if (nw) {
        visit[v] = vis | nw;
        ++newly;
        ndeg += (uint64_t)(out_rows[v + 1] - out_rows[v]);
      }
    }
    ms_count_sources(nw, cnt);
  }
  if (has_wide) {
    const int64_t nv = (int64_t)wd.cnt[0];
    for (int64_t base = wave << 6; base < nv; base += nwaves << 6) {
      const int64_t k = base + lane;
      uint64_t nw = 0;
      if (k < nv) {
        const int v = wd.v[k];
        const uint64_t vis = visit[v];
        nw = wd.acc[k] & all & ~vis;
        if (nw) {
          wd.acc[k] = 0ull;
          visit[v] = vis | nw;
          ++newly;
          ndeg += (uint64_t)(out_rows[v + 1] - out_rows[v]);
        }
        next[v] = nw;
      }
      ms_count_sources(nw, cnt);
    }
  }
  ms_flush(c, newly, ndeg, cnt);
}

// One edge of a top-down level: next[u] |= f & ~visit[u].
__device__ __forceinline__ void ms_visit(uint64_t f, int32_t u, const uint64_t *visit,
                                         uint64_t *next) {
  const uint64_t b = f & ~visit[u];
  if (b && (next[u] & b) != b)
    atomicOr((unsigned long long *)&next[u], (unsigned long long)b);
}

// Top-down level, scatter part: next[u] |= front[v] & ~visit[u]; the edges of
// wide rows (has_wide) chunk by chunk, one wavefront each.
__global__ void __launch_bounds__(BLOCK)
    k_msbfs_push(const int64_t *__restrict__ rows,
                 const int32_t *__restrict__ cols, int64_t n,
                 const uint64_t *__restrict__ visit,
                 const uint64_t *__restrict__ front, uint64_t *next, bool has_wide,
                 ms_wide_t wd) {
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> LOG_WAVE;
  for (int64_t base = wave << 6; base < n; base += nwaves << 6) {
    const int64_t v = base + lane;
    const uint64_t f = (v < n) ? front[v] : 0ull;
    if (!f) continue;
    const int64_t s = rows[v], e = rows[v + 1];
    if (e - s > MS_WIDE) continue;
    for (int64_t j = s; j < e; ++j) ms_visit(f, cols[j], visit, next);
  }
  if (!has_wide) return;
  const int64_t ne = (int64_t)wd.cnt[1];
  for (int64_t i = wave; i < ne; i += nwaves) {
    const int2 e = wd.ent[i];
    const int v = wd.v[e.x];
    const uint64_t f = front[v];
    if (!f) continue;
    const int64_t s = rows[v] + (int64_t)e.y * MS_CHUNK;
    const int64_t end = MIN(rows[v + 1], s + MS_CHUNK);
    for (int64_t j = s + lane; j < end; j += WAVE) ms_visit(f, cols[j], visit, next);
  }
}

// First top-down level: the frontier is the sources, which are often the
// graph's hubs, so their edges are spread evenly over the whole grid (edge k
// of the sources' concatenated lists, found by binary search over their
// degree prefix) instead of one wavefront per source vertex.
struct ms_seeds_t {
  int nsrc;
  int32_t src[64];
  int64_t pre[65];  // exclusive prefix of the sources' degrees
};

__global__ void __launch_bounds__(BLOCK)
    k_msbfs_push_seeds(const int64_t *__restrict__ rows,
                       const int32_t *__restrict__ cols,
                       const uint64_t *__restrict__ visit,
                       const uint64_t *__restrict__ front, uint64_t *next,
                       ms_seeds_t sd) {
  __shared__ int64_t s_pre[65];
  __shared__ int64_t s_row[64];
  __shared__ uint64_t s_bits[64];
  const int t = threadIdx.x;
  if (t <= sd.nsrc) s_pre[t] = sd.pre[t];
  if (t < sd.nsrc) {
    s_row[t] = rows[sd.src[t]];
    s_bits[t] = front[sd.src[t]];
  }
  __syncthreads();
  const int64_t total = s_pre[sd.nsrc];
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + t; k < total; k += stride) {
    int lo = 0, hi = sd.nsrc;  // the last source with s_pre[lo] <= k
    while (hi - lo > 1) {
      const int mid = (lo + hi) >> 1;
      if (s_pre[mid] <= k)
        lo = mid;
      else
        hi = mid;
    }
    ms_visit(s_bits[lo], cols[s_row[lo] + (k - s_pre[lo])], visit, next);
  }
}

// Top-down level, sweep part: keep only new bits, fold them into visit.
__global__ void __launch_bounds__(BLOCK)
    k_msbfs_sweep(const int64_t *__restrict__ rows, int64_t n,
                  uint64_t *__restrict__ visit, uint64_t *__restrict__ next,
                  ms_counters_t *c) {
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> LOG_WAVE;
  unsigned long long newly = 0, ndeg = 0, cnt = 0;
  for (int64_t base = wave << 6; base < n; base += nwaves << 6) {
    const int64_t v = base + lane_id();
    uint64_t nw = 0;
    if (v < n) {
      const uint64_t x = next[v];
      if (x) {
        const uint64_t vis = visit[v];
        nw = x & ~vis;
        next[v] = nw;
        if (nw) {
          visit[v] = vis | nw;
          ++newly;
          ndeg += (uint64_t)(rows[v + 1] - rows[v]);
        }
      }
    }
    ms_count_sources(nw, cnt);
  }
  ms_flush(c, newly, ndeg, cnt);
}

// End of a level, one workgroup: the slots' sum to `out` (pinned host
// memory), then its mark; the slots cleared for the next level.
constexpr int MS_COUNTS = 66;  // newly, newly_deg, per_src
constexpr int MS_MARK = 72;    // (in the padding of a slot)
__global__ void __launch_bounds__(BLOCK)
    k_msbfs_finish(ms_counters_t *c, unsigned long long *out, unsigned long long seq) {
  __shared__ unsigned long long sh[BLOCK / WAVE][WAVE + 2];
  static_assert(sizeof(ms_counters_t) % 8 == 0, "slots of whole words");
  constexpr int NW = BLOCK / WAVE, W = sizeof(ms_counters_t) / 8;
  const int w = threadIdx.x >> LOG_WAVE, lane = lane_id();
  unsigned long long *p = (unsigned long long *)c;
  for (int k = lane; k < MS_COUNTS; k += WAVE) {
    unsigned long long t = 0;
#pragma unroll
    for (int i = 0; i < MS_SLOTS / NW; ++i) {
      t += p[(w + i * NW) * W + k];
      p[(w + i * NW) * W + k] = 0ull;
    }
    sh[w][k] = t;
  }
  __syncthreads();
  if (threadIdx.x < MS_COUNTS) {
    unsigned long long t = 0;
#pragma unroll
    for (int i = 0; i < NW; ++i) t += sh[i][threadIdx.x];
    out[threadIdx.x] = t;
    __threadfence_system();
  }
  __syncthreads();
  if (threadIdx.x == 0) publish(out + MS_MARK, seq);
}

__global__ void __launch_bounds__(BLOCK)
    k_msbfs_seed(uint64_t *visit, uint64_t *front, const int32_t *src,
                 int nsrc) {
  const int s = threadIdx.x;
  if (s < nsrc) {
    atomicOr((unsigned long long *)&visit[src[s]], 1ull << s);
    atomicOr((unsigned long long *)&front[src[s]], 1ull << s);
  }
}

}  // namespace gsw
