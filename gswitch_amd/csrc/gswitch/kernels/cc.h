// Connected components by tree hooking over the CSR, with subgraph sampling
// (Afforest: Sutton, Ben-Nun, Bar-Noy, "Optimizing Parallel Graph
// Connectivity Computation via Subgraph Sampling", IPDPS 2018).
//
// p[v] is a parent pointer with p[v] <= v; roots have p[r] = r. link(u, v)
// hooks the larger of the two roots under the smaller one with a
// compare-and-swap, so every tree's root is the smallest id in it and, once a
// component is one tree, its root is the component's minimum vertex id: the
// canonical label of the reference's CC (application/cc.cu:34-66). link
// never waits on another lane: each failed CAS means the root it tried moved
// to a smaller value, so the loop ends.
//
// Phases (a fixed sequence of launches, no host decisions in between, so it
// can live in a captured graph):
//  1. start: every vertex hooks under a smaller vertex it reaches over first
//     (smallest) in-neighbours, with a plain store (k_cc_start), compress;
//  2. sampling: every vertex links its second neighbour (or its only one,
//     where that is larger), compress;
//  3. skip set S: vertices whose root is a chosen root -- the most frequent
//     root of a vertex sample for one graph, or each instance's first vertex
//     (its smallest id) for a disjoint batch. Vertices outside S link all
//     their edges; a vertex in S skips the edges that stay inside its
//     instance (their other end is either in the same tree already or
//     outside S, and then links the edge itself) and links only edges that
//     leave its instance, so a batch whose instances share edges stays
//     correct;
//  4. compress: p[v] = root(v).
// Undirected graphs only use S (an edge must be visible from both ends);
// a directed graph links every out-edge of every vertex (weak components).
#pragma once
#include "../utils/runtime.h"
#include "../utils/wave.h"

namespace gsw {

constexpr int CC_WIDE = 128;  // degree above which a wavefront shares a row

constexpr int CC_HALVE_AFTER = 16;  // steps of a link before it halves its path
constexpr int CC_HOPS = 4;          // first neighbours a vertex follows at the start
constexpr int CC_SILP = 4;          // vertices a lane samples at once

// A parent pointer, possibly an old one from this XCD's L2: every value that an
// entry ever holds is an ancestor of its vertex, so an old one is too (a store
// that halves a path may even put a larger ancestor back), and a hooked vertex
// that still looks like a root fails its CAS.
// (Loads that are coherent over the device cost more: 2 M-vertex random graph
// of mean degree 6, whole CC 276 against 303 us.)
__device__ __forceinline__ int cc_get(const int *p, int64_t i) {
  return __hip_atomic_load(p + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Join the trees of u and v: hook the larger root under the smaller one with
// a CAS, walking up from the parents (two steps at a time on the larger side)
// while neither is a root. The larger side strictly decreases: a vertex that
// an old pointer shows as a root fails its CAS, which returns its parent.
// A link that has walked CC_HALVE_AFTER steps halves its path as it goes on:
// on a grid the trees of the start are strips whose links chain up over
// thousands of strips (3000 x 2851 grid: this pass 1.9 ms without halving,
// 0.47 ms with it), while on random graphs and R-MAT walks are short and the
// stores of halving at once cost more than they save (the random graph above:
// after 2 steps 1110 us, after 8 370, after 16 or never 277).
// Lanes of a wavefront at one apparent root send one CAS: with one each, every
// lane that still sees a hooked root as a root queues an atomic on it (two hubs
// over the same 262 K leaves: 2000 us, so 111; R-MAT 20 with half its edges,
// directed: the second neighbours' links 406 us). Returns an ancestor of both,
// near the root, for the next link of a row.
__device__ __forceinline__ int cc_link(int a, int b, int *p) {
  for (int step = 0; a != b; ++step) {
    const int hi = a > b ? a : b, lo = a > b ? b : a;
    int ph = cc_get(p, hi);
    if (ph == lo) return lo;
    if (ph == hi) {
      // the lanes at the first lane's root go on from where its leader found
      // or hooked that root
      const int h0 = __builtin_amdgcn_readfirstlane(hi);
      const int leader = __builtin_ctzll(ballot(hi == h0));
      const bool mine = hi != h0 || lane_id() == leader;
      int old = hi;
      if (mine) old = atomicCAS(p + hi, hi, lo);
      const int o0 = readlane(old, leader), l0 = readlane(lo, leader);
      if (mine) {
        ph = old;
        if (ph == hi) return lo;
      } else {
        ph = o0 == hi ? l0 : o0;
        if (ph == lo) return lo;
      }
    }
    a = cc_get(p, ph);
    if (step >= CC_HALVE_AFTER)
      __hip_atomic_store(p + hi, a, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    b = cc_get(p, lo);
  }
  return a;
}

// Where v hooks at the start: the smallest vertex within CC_HOPS steps over
// first (smallest) in-neighbours, each smaller than the one before.
__device__ __forceinline__ int cc_start_of(int v, const int32_t *__restrict__ first) {
  int x = v;
  for (int h = 0; h < CC_HOPS; ++h) {
    const int y = first[x];
    if (y < 0 || y >= x) break;
    x = y;
  }
  return x;
}

// p[v] <- a smaller vertex of v's component, or v. Plain stores: no two lanes
// write one entry, and entries are only read by later launches. (Against an
// identity fill and a CAS link of every first neighbour, and with k_cc_mode
// below: CC of R-MAT 21 on the device 180 -> 73 us. Following up to 8 or 32 neighbours only shortens
// chains that the compress shortens faster.)
__global__ void __launch_bounds__(BLOCK)
    k_cc_start(const int32_t *__restrict__ first, int *__restrict__ p, int64_t n) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * blockDim.x)
    p[v] = cc_start_of((int)v, first);
}

// Link every vertex with its second neighbour, or with its only one where that
// is larger, so that k_cc_start did not hook it (with `skip_lv`, only the
// vertices whose skip_lv entry is negative). Without the latter a star whose
// hub has the largest id was left to k_cc_rest, where one wavefront walked the
// hub: 1 M leaves 11.1 ms, now 0.04.
__global__ void __launch_bounds__(BLOCK)
    k_cc_sample(const int64_t *__restrict__ rows, const int32_t *__restrict__ cols,
                int64_t n, int *p, const int *__restrict__ skip_lv) {
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (int64_t v0 = tid; v0 < n; v0 += stride * CC_SILP) {
    // the vertices' loads together, then their links one after another
    // (2 M-vertex random graph, R-MAT 21 of edge factor 4 with shuffled ids:
    // whole CC 277 -> 257 and 223 -> 180 us against one vertex at a time)
    int a[CC_SILP], b[CC_SILP];
    int64_t s[CC_SILP];
    bool only[CC_SILP];
#pragma unroll
    for (int k = 0; k < CC_SILP; ++k) {
      const int64_t v = v0 + k * stride;
      s[k] = -1;
      only[k] = false;
      if (v < n && !(skip_lv && skip_lv[v] >= 0)) {
        const int64_t r = rows[v], e = rows[v + 1];
        only[k] = e - r == 1;
        if (e > r) s[k] = only[k] ? r : r + 1;
      }
    }
#pragma unroll
    for (int k = 0; k < CC_SILP; ++k) a[k] = s[k] >= 0 ? cols[s[k]] : 0;
#pragma unroll
    for (int k = 0; k < CC_SILP; ++k) {
      const int64_t v = v0 + k * stride;
      b[k] = a[k];
      if (s[k] >= 0 && !(only[k] && a[k] < v)) {
        a[k] = cc_get(p, a[k]);
        b[k] = cc_get(p, v);
      }
    }
#pragma unroll
    for (int k = 0; k < CC_SILP; ++k) (void)cc_link(a[k], b[k], p);
  }
}

// p[v] <- root of v (no links run meanwhile, so p is a forest whose roots
// stay put). Every vertex moves its own pointer to its grandparent until
// the parent is a root; the pointers it reads are being shortened by their
// own vertices at the same time, so a chain of length d collapses in about
// log d steps per vertex instead of each vertex walking it alone. Random
// loads beyond the L2 bound it (several vertices per lane at once: no faster).
__global__ void __launch_bounds__(BLOCK) k_cc_compress(int *p, int64_t n) {
  for (int64_t v = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; v < n;
       v += (int64_t)gridDim.x * blockDim.x) {
    int x = cc_get(p, v);
    int y = cc_get(p, x);
    while (y != x) {
      __hip_atomic_store(p + v, y, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      x = y;
      y = cc_get(p, x);
    }
  }
}

// ---- choosing the skipped component on the device ------------------------
// The most frequent root among a fixed sample of vertices (ids from a
// SplitMix64 output mix over key + (i+1)*phi, scaled to [0, n) by a
// multiply-high: the host generators' counter RNG). No host read, so the
// whole CC is one asynchronous launch sequence.
constexpr int CC_MAX_SAMPLES = 4096;
constexpr int CC_MODE_BLOCK = 1024;
constexpr int CC_MODE_SLOTS = 6144;  // open addressing, at most 2/3 full
constexpr uint64_t CC_SAMPLE_KEY = 0xCC5A3D1Eull;

__device__ __forceinline__ uint64_t cc_mix64(uint64_t z) {
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// *skip <- the most frequent root of the k sampled vertices (ties: the
// smallest). One workgroup, 1 <= k <= CC_MAX_SAMPLES: the roots are counted in
// an LDS hash table, equal roots of a wavefront by one atomic (most samples
// hit the large component), then a 64-bit max of (count, INT_MAX - root) over
// the table picks the winner. (Latency of one workgroup bounds it; a bitonic
// sort of the samples and serial run counts took 61-88 us for 1024 samples.)
__global__ void __launch_bounds__(CC_MODE_BLOCK)
    k_cc_mode(const int *p, int k, int64_t n, int *skip) {
  __shared__ int s_key[CC_MODE_SLOTS], s_cnt[CC_MODE_SLOTS];
  __shared__ unsigned long long best;
  for (int i = threadIdx.x; i < CC_MODE_SLOTS; i += blockDim.x) {
    s_key[i] = -1;
    s_cnt[i] = 0;
  }
  if (threadIdx.x == 0) best = 0;
  __syncthreads();
  const uint64_t key = cc_mix64(cc_mix64(CC_SAMPLE_KEY));
  for (int i0 = threadIdx.x & ~(WAVE - 1); i0 < k; i0 += blockDim.x) {
    const int i = i0 + lane_id();
    int x = -1;
    if (i < k) {
      const uint64_t r = cc_mix64(key + (uint64_t)(i + 1) * 0x9E3779B97F4A7C15ull);
      x = cc_get(p, (int64_t)__umul64hi(r, (uint64_t)n));
    }
    uint64_t todo = ballot(i < k);
    while (todo) {
      // the first open lane counts every lane with its root
      const int lead = __builtin_ctzll(todo);
      const int y = readlane(x, lead);
      const uint64_t same = ballot(x == y) & todo;
      todo &= ~same;
      if (lane_id() == lead) {
        int h = (int)(((uint32_t)y * 2654435761u) % CC_MODE_SLOTS);
        for (;;) {
          const int old = atomicCAS(&s_key[h], -1, y);
          if (old == -1 || old == y) break;
          h = h + 1 == CC_MODE_SLOTS ? 0 : h + 1;
        }
        atomicAdd(&s_cnt[h], __popcll(same));
      }
    }
  }
  __syncthreads();
  unsigned long long top = 0;
  for (int i = threadIdx.x; i < CC_MODE_SLOTS; i += blockDim.x)
    if (s_cnt[i]) {
      const unsigned long long c =
          ((unsigned long long)s_cnt[i] << 32) | (unsigned)(INT_MAX - s_key[i]);
      top = c > top ? c : top;
    }
  top = wave_max_any(top);
  if (lane_id() == 0 && top) atomicMax(&best, top);
  __syncthreads();
  if (threadIdx.x == 0) *skip = INT_MAX - (int)(unsigned)(best & 0xFFFFFFFFull);
}

// Instance of v: the largest i with offsets[i] <= v (offsets ascending,
// offsets[0] = 0, count + 1 entries).
__device__ __forceinline__ int64_t cc_instance(const int64_t *off, int64_t count,
                                               int64_t v) {
  int64_t lo = 0, hi = count;
  while (hi - lo > 1) {
    const int64_t mid = (lo + hi) >> 1;
    if (off[mid] <= v)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

// Instance of vertex v of a wavefront whose lanes hold base .. base + 63:
// one search for base (every lane the same addresses), then forward steps.
__device__ __forceinline__ int64_t cc_instance_wave(const int64_t *off, int64_t count,
                                                    int64_t base, int64_t v) {
  int64_t i = cc_instance(off, count, base);
  while (i + 1 < count && off[i + 1] <= v) ++i;
  return i;
}

// For a batch of instances whose edges stay inside their instance (checked
// by k_cc_cross) and BFS levels from every instance's first vertex: the
// vertices the BFS reached form the component of that first vertex, the
// smallest id of the instance, so that id is their label; every other
// vertex starts as in k_cc_start (its in-neighbours are unreached as well).
__global__ void __launch_bounds__(BLOCK)
    k_cc_seed_levels(int *p, const int *__restrict__ lv, const int32_t *__restrict__ first,
                     const int64_t *__restrict__ off, int64_t count, int64_t n) {
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> LOG_WAVE;
  for (int64_t base = wave << 6; base < n; base += nwaves << 6) {
    const int64_t v = base + lane;
    if (v < n)
      p[v] = lv[v] >= 0 ? (int)off[cc_instance_wave(off, count, base, v)]
                        : cc_start_of((int)v, first);
  }
}

// *flag = 1 if an edge leaves its source's instance.
__global__ void __launch_bounds__(BLOCK)
    k_cc_cross(const int64_t *__restrict__ rows, const int32_t *__restrict__ cols,
               int64_t n, const int64_t *__restrict__ off, int64_t count, int *flag) {
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> LOG_WAVE;
  bool out = false;
  for (int64_t base = wave << 6; base < n; base += nwaves << 6) {
    const int64_t v = base + lane;
    int64_t s = 0, e = 0, lo = 0, hi = 0;
    if (v < n) {
      s = rows[v];
      e = rows[v + 1];
      const int64_t i = cc_instance_wave(off, count, base, v);
      lo = off[i];
      hi = off[i + 1];
    }
    // columns of a row are sorted: its first and last entries decide
    if (e > s && (cols[s] < lo || cols[e - 1] >= hi)) out = true;
  }
  if (ballot(out) && lane == 0) atomicOr(flag, 1);
}

// Phase 3. skip_root >= 0: S = {v : p[v] == skip_root} (one graph);
// skip_root == -1: S = {v : p[v] == first vertex of v's instance} with
// `off` the count + 1 instance offsets; skip_root == -2: no skipping. A
// non-null skip_dev replaces skip_root by *skip_dev (written by k_cc_mode).
// (Every edge of a row: its first one is hooked only where k_cc_start found
// its other end smaller.)
// One wavefront per 64 vertices; rows longer than CC_WIDE are walked by
// the whole wavefront, one at a time. `disjoint`: no edge leaves an
// instance (skip_root == -1), so a vertex of S links nothing.
__global__ void __launch_bounds__(BLOCK)
    k_cc_rest(const int64_t *__restrict__ rows, const int32_t *__restrict__ cols,
              int64_t n, int skip_arg, const int *skip_dev,
              const int64_t *__restrict__ off, int64_t count, int *p,
              int disjoint) {
  const int skip_root = skip_dev ? *skip_dev : skip_arg;
  const int lane = lane_id();
  const int64_t wave = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) >> LOG_WAVE;
  const int64_t nwaves = ((int64_t)gridDim.x * blockDim.x) >> LOG_WAVE;
  for (int64_t base = wave << 6; base < n; base += nwaves << 6) {
    const int64_t v = base + lane;
    int64_t s = 0, e = 0, lo = 0, hi = 0;
    bool in_s = false;
    int root = 0;
    if (v < n) {
      s = rows[v];
      e = rows[v + 1];
      root = cc_get(p, v);
      if (skip_root >= 0) {
        in_s = root == skip_root;
        hi = n;
      } else if (skip_root == -1) {
        const int64_t i = cc_instance(off, count, v);
        lo = off[i];
        hi = off[i + 1];
        in_s = root == (int)lo;
      }
      // one graph, or instances with no edge between them: a vertex of S
      // has nothing to link
      if (in_s && (skip_root >= 0 || disjoint)) e = s;
    }
    const bool wide = (e - s) > CC_WIDE;
    if (!wide)
      for (int64_t j = s; j < e; ++j) {
        const int u = cols[j];
        if (!in_s || u < lo || u >= hi) root = cc_link(root, cc_get(p, u), p);
      }
    uint64_t wmask = ballot(wide);
    while (wmask) {
      const int w = __builtin_ctzll(wmask);
      wmask &= wmask - 1;
      const int64_t ws = __shfl(s, w, 64), we = __shfl(e, w, 64);
      const int64_t wl = __shfl(lo, w, 64), wh = __shfl(hi, w, 64);
      const bool wi = __shfl((int)in_s, w, 64) != 0;
      int wr = __shfl(root, w, 64);
      // (the next column is loaded before this one's link: a directed hub of
      // 1 M edges 18.7 -> 15.8 ms)
      int64_t j = ws + lane;
      int next = j < we ? cols[j] : 0;
      for (; j < we; j += WAVE) {
        const int u = next;
        if (j + WAVE < we) next = cols[j + WAVE];
        if (!wi || u < wl || u >= wh) wr = cc_link(wr, cc_get(p, u), p);
      }
    }
  }
}

}  // namespace gsw
