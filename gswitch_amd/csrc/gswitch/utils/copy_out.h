// Results to the caller's (pageable) host memory.
//
// A plain device-to-host hipMemcpy into pageable memory moves one MiB at a
// time: copy into the runtime's pinned buffer, wait, copy on to the caller by
// one thread (on MI355X 20 + 65 us per MiB, 11 GB/s), so it costs more than
// most traversals. Here a kernel stores the array into a pinned ring piece by
// piece and marks every finished piece in host memory, and worker threads copy
// a piece on as soon as its mark is there: the link (56 GB/s) and the host
// copies overlap, with one launch per 4 MiB and no wait on the stream at all:
// 16.8 MB 980 -> 390 us, 8.4 MB 480 -> 215, 4.2 MB 243 -> 132, 64 KB 35 -> 15
// (the caller's buffer warm; 67 MB into new pages 6.5 -> 2.0 ms).
// (Pinned copies by hipMemcpyAsync with an event each were no faster than the
// plain copy up to 8 MB: about 30 us of overhead per copy.)
#pragma once
#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <initializer_list>
#include <mutex>
#include <thread>
#include <vector>

#include "runtime.h"

namespace gsw {

constexpr size_t OUT_PIECE = 32 << 10;          // bytes per mark
constexpr size_t OUT_HALF = 4 << 20;            // bytes per launch: half the ring
constexpr int OUT_PIECES = OUT_HALF / OUT_PIECE;
constexpr int OUT_GRID = 32;   // workgroups: pieces finish in order, link full
constexpr int OUT_MARK = 16;   // uint32 per mark (one 64-byte line)

// Pieces of [src, src + bytes) to dst (pinned host memory), piece p's mark to
// `seq` once it is there.
__global__ void __launch_bounds__(BLOCK)
    k_copy_out(const char *__restrict__ src, char *dst, int64_t bytes, uint32_t *marks,
               uint32_t seq) {
  const int64_t np = (bytes + (int64_t)OUT_PIECE - 1) / (int64_t)OUT_PIECE;
  const bool wide = (((uintptr_t)src | (uintptr_t)dst) & 15) == 0;
  const bool words = (((uintptr_t)src | (uintptr_t)dst) & 3) == 0;
  for (int64_t p = blockIdx.x; p < np; p += gridDim.x) {
    const int64_t lo = p * (int64_t)OUT_PIECE;
    const int64_t hi = MIN(bytes, lo + (int64_t)OUT_PIECE);
    int64_t at = lo;
    if (wide) {
      const int64_t n = (hi - at) / 16;
      const uint4 *s = (const uint4 *)(src + at);
      uint4 *d = (uint4 *)(dst + at);
      for (int64_t i = threadIdx.x; i < n; i += BLOCK) d[i] = s[i];
      at += n * 16;
    }
    if (words) {
      const int64_t n = (hi - at) / 4;
      const uint32_t *s = (const uint32_t *)(src + at);
      uint32_t *d = (uint32_t *)(dst + at);
      for (int64_t i = threadIdx.x; i < n; i += BLOCK) d[i] = s[i];
      at += n * 4;
    }
    for (int64_t i = at + threadIdx.x; i < hi; i += BLOCK) dst[i] = src[i];
    __threadfence_system();  // this thread's stores before the mark below
    __syncthreads();
    if (threadIdx.x == 0)
      __hip_atomic_store(marks + p * OUT_MARK, seq, __ATOMIC_RELEASE,
                         __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

// A pinned ring of `cap` bytes, at most two halves of OUT_HALF (smaller where
// only small results were asked for: pinning takes time by the page), and its
// marks.
struct out_ring_t {
  int dev = -1;
  size_t cap = 0;
  char *buf = nullptr;
  uint32_t *marks = nullptr;
  uint32_t seq = 0;  // of the last launch
  void build(int d, size_t bytes) {
    dev = d;
    cap = bytes;
    const size_t mb = sizeof(uint32_t) * 2 * OUT_PIECES * OUT_MARK;
    H_ERR(hipHostMalloc((void **)&buf, cap));
    H_ERR(hipHostMalloc((void **)&marks, mb));
    std::memset(marks, 0, mb);
  }
  void release() {
    if (buf) (void)hipHostFree(buf);
    if (marks) (void)hipHostFree(marks);
    buf = nullptr;
    marks = nullptr;
  }
};

// Rings shared by every graph handle of the process (pinning one costs more
// than filling it). A ring belongs to one call from take() to give(), so
// calls on different threads, streams and devices do not share one. A device
// keeps as many as calls have been under way on it at once, KEEP at most, and
// none once the last handle is gone. (With two kept in the whole process, every
// third call at once pinned its ring anew: labels of R-MAT 18 on 8 threads 60 us
// per call, now 42.)
struct out_pool_t {
  static constexpr size_t KEEP = 8;
  struct use_t {
    int dev = -1;
    size_t now = 0, most = 0;  // calls under way
    std::vector<out_ring_t> idle;
  };
  std::mutex mu;
  std::vector<use_t> uses;  // one per device
  int64_t handles = 0;

  use_t &of(int dev) {
    for (use_t &u : uses)
      if (u.dev == dev) return u;
    uses.emplace_back();
    uses.back().dev = dev;
    uses.back().idle.reserve(KEEP);
    return uses.back();
  }

  // a ring of at least `need` bytes; an idle one that is too small goes
  out_ring_t take(int dev, size_t need) {
    out_ring_t small;
    {
      std::lock_guard<std::mutex> lock(mu);
      use_t &u = of(dev);
      u.most = std::max(u.most, ++u.now);
      for (size_t i = u.idle.size(); i-- > 0;)
        if (u.idle[i].cap >= need) {
          const out_ring_t r = u.idle[i];
          u.idle[i] = u.idle.back();
          u.idle.pop_back();
          return r;
        }
      if (!u.idle.empty()) {
        small = u.idle.back();
        u.idle.pop_back();
      }
    }
    small.release();
    out_ring_t r;
    size_t cap = 2 * OUT_PIECE;
    while (cap < need) cap *= 2;
    try {
      r.build(dev, cap);
    } catch (...) {
      r.release();
      std::lock_guard<std::mutex> lock(mu);
      --of(dev).now;
      throw;
    }
    return r;
  }
  void give(out_ring_t r) {
    {
      std::lock_guard<std::mutex> lock(mu);
      use_t &u = of(r.dev);
      --u.now;
      if (handles > 0 && u.idle.size() + u.now < std::min(u.most, KEEP)) {
        u.idle.push_back(r);
        return;
      }
    }
    r.release();
  }
  void handle_made() {
    std::lock_guard<std::mutex> lock(mu);
    ++handles;
  }
  void handle_gone() {
    std::vector<out_ring_t> dead;
    {
      std::lock_guard<std::mutex> lock(mu);
      if (--handles == 0)
        for (use_t &u : uses) {
          dead.insert(dead.end(), u.idle.begin(), u.idle.end());
          u.idle.clear();
          u.most = u.now;
        }
    }
    for (out_ring_t &r : dead) r.release();
  }
};

inline out_pool_t &out_pool() {
  // never destroyed: the runtime may be gone before static destructors run
  static out_pool_t *pool = new out_pool_t;
  return *pool;
}
struct out_ref_t {
  out_ref_t() { out_pool().handle_made(); }
  ~out_ref_t() { out_pool().handle_gone(); }
  out_ref_t(const out_ref_t &) = delete;
  out_ref_t &operator=(const out_ref_t &) = delete;
};

// A result array: `bytes` from device memory to host memory.
struct out_t {
  void *dst;
  const void *src;
  size_t bytes;
};

class copy_out_t {
  // at most OUT_HALF bytes of one array: one launch, into a place of its own
  // in the ring where everything fits, else into half (index & 1)
  struct part_t {
    char *dst;
    const char *src;
    size_t bytes;
    size_t first;  // its first piece
    size_t slot;   // its first piece's place in the ring
  };
  bool packed = false;
  std::vector<part_t> parts;
  size_t n_pieces = 0;
  std::vector<std::atomic<size_t>> left;  // pieces of a part not copied on yet
  std::vector<uint32_t> seqs;
  std::atomic<size_t> next{0}, launched{0};  // pieces taken; parts launched
  std::atomic<bool> failed{false};
  std::mutex mu;
  std::exception_ptr error;
  int dev = 0;
  hipStream_t st = nullptr;
  out_ring_t ring;

  static size_t pieces_of(size_t bytes) { return (bytes + OUT_PIECE - 1) / OUT_PIECE; }

  // part k, once its place in the ring is free; called by one thread at a
  // time, in order
  void launch(size_t k) {
    const part_t &q = parts[k];
    if (++ring.seq == 0) ring.seq = 1;
    seqs[k] = ring.seq;
    const int grid = (int)std::min<size_t>(OUT_GRID, pieces_of(q.bytes));
    hipLaunchKernelGGL(k_copy_out, dim3(grid), dim3(BLOCK), 0, st, q.src,
                       ring.buf + q.slot * OUT_PIECE, (int64_t)q.bytes,
                       ring.marks + q.slot * OUT_MARK, ring.seq);
    H_ERR(hipGetLastError());
    launched.store(k + 1, std::memory_order_release);
  }

  void pause() const { __builtin_ia32_pause(); }

  // until piece i of part k is in the ring; false if another worker failed
  bool await(size_t k, size_t i) {
    while (launched.load(std::memory_order_acquire) <= k) {
      if (failed) return false;
      pause();
    }
    const uint32_t *mark = ring.marks + (parts[k].slot + i) * OUT_MARK;
    for (int64_t spin = 1; __atomic_load_n(mark, __ATOMIC_ACQUIRE) != seqs[k]; ++spin) {
      if (failed) return false;
      pause();
      if (spin % 65536 == 0) {
        // a stream that failed, or ended without the mark, never sets it
        const hipError_t e = hipStreamQuery(st);
        if (e == hipErrorNotReady) continue;
        H_ERR(e);
        GSW_REQUIRE(__atomic_load_n(mark, __ATOMIC_ACQUIRE) == seqs[k], E_HIP,
                    "result copy did not arrive");
      }
    }
    return true;
  }

  void work() noexcept {
    try {
      H_ERR(hipSetDevice(dev));
      size_t k = 0;
      for (;;) {
        const size_t i = next.fetch_add(1);
        if (i >= n_pieces || failed) return;
        while (k + 1 < parts.size() && i >= parts[k + 1].first) ++k;
        const size_t at = i - parts[k].first;
        if (!await(k, at)) return;
        const size_t b = at * OUT_PIECE;
        std::memcpy(parts[k].dst + b, ring.buf + parts[k].slot * OUT_PIECE + b,
                    std::min(OUT_PIECE, parts[k].bytes - b));
        // the worker that empties a half refills it (parts are emptied in
        // order: part k + 1 is launched, its predecessor's half is this one)
        if (left[k].fetch_sub(1, std::memory_order_acq_rel) == 1 && k + 2 < parts.size()) {
          std::lock_guard<std::mutex> lock(mu);
          refill();
        }
      }
    } catch (...) {
      std::lock_guard<std::mutex> lock(mu);
      if (!error) error = std::current_exception();
      failed = true;
    }
  }

  // launch every part whose half is free (under mu)
  void refill() {
    for (size_t k = launched; k < parts.size(); ++k) {
      if (!packed && k >= 2 && left[k - 2].load(std::memory_order_acquire) != 0) return;
      launch(k);
    }
  }

 public:
  // Copies every array with a destination; returns when the data is there.
  void run(std::initializer_list<out_t> outs) {
    H_ERR(hipGetDevice(&dev));
    st = stream();
    size_t total = 0;
    for (const out_t &o : outs) {
      if (!o.dst || o.bytes == 0) continue;
      // memory the runtime knows (pinned, managed, device): one direct copy
      hipPointerAttribute_t attr;
      const hipError_t e = hipPointerGetAttributes(&attr, o.dst);
      if (e != hipSuccess) (void)hipGetLastError();  // clear the failed query
      if (e == hipSuccess && attr.type != hipMemoryTypeUnregistered) {
        H_ERR(hipMemcpyAsync(o.dst, o.src, o.bytes, hipMemcpyDefault, st));
        H_ERR(hipStreamSynchronize(st));
        continue;
      }
      total += o.bytes;
      for (size_t b = 0; b < o.bytes; b += OUT_HALF) {
        const size_t len = std::min(OUT_HALF, o.bytes - b);
        parts.push_back({(char *)o.dst + b, (const char *)o.src + b, len, n_pieces, 0});
        n_pieces += pieces_of(len);
      }
    }
    if (total == 0) return;
    left = std::vector<std::atomic<size_t>>(parts.size());
    for (size_t k = 0; k < parts.size(); ++k) left[k] = pieces_of(parts[k].bytes);
    seqs.resize(parts.size());
    packed = n_pieces <= 2 * OUT_PIECES;
    for (size_t k = 0; k < parts.size(); ++k)
      parts[k].slot = packed ? parts[k].first : (k & 1) * OUT_PIECES;
    ring = out_pool().take(dev, packed ? n_pieces * OUT_PIECE : 2 * OUT_HALF);
    std::vector<std::thread> th;
    try {
      std::lock_guard<std::mutex> lock(mu);
      refill();
    } catch (...) {
      error = std::current_exception();
      failed = true;
    }
    if (!failed) {
      // helpers from 2 MiB on (a thread starts in about 20 us), three until
      // the caller's pages outlast the link (they fault in as they are filled)
      const unsigned cpus = std::max(1u, std::thread::hardware_concurrency());
      const size_t most = total >= ((size_t)32 << 20) ? 6 : 3;
      const size_t helpers = total < ((size_t)2 << 20)
                                 ? 0
                                 : std::min<size_t>({total >> 20, most, (size_t)cpus - 1});
      try {
        th.reserve(helpers);
        for (size_t i = 0; i < helpers; ++i) th.emplace_back([this] { work(); });
      } catch (...) {
        // fewer workers: the others take every piece
      }
      work();
    }
    for (std::thread &t : th) t.join();
    // (launches of a failed call may still write the ring)
    if (failed) (void)hipStreamSynchronize(st);
    out_pool().give(ring);
    if (error) std::rethrow_exception(error);
  }
};

// Device arrays to the caller's host arrays (null destinations are skipped),
// ordered after the engine's stream.
inline void copy_out(std::initializer_list<out_t> outs) { copy_out_t().run(outs); }

}  // namespace gsw
