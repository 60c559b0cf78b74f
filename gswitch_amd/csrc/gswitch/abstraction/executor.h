// executor_t: frontier generation and expand dispatch.
//
// filter() follows executor_t::filter + __filter (src/abstraction/
// executor.cuh:21-72, src/kernel_libs/filter.cuh:197-252): set the frontier
// format, compact bitmap -> queue when a queue is needed and it was not
// produced by a fused expand, swap the queues, size the grid and run the
// fusion compensation pass. expand() follows executor_t::expand
// (executor.cuh:74-148): one launch of the chosen {direction, LB, fusion}
// variant, timing history, and the fused -> standalone fallback when an
// expand takes more than 5x the average.
//
// Host<->device traffic per level: standalone levels wait once (the
// inspector's counters); fused levels wait once after the expand (the next
// queue's length, which also tells convergence), those of run_ahead() once per
// batch of up to eight. Queue lengths are otherwise known on the host from the
// inspector's counts.
#pragma once
#include <cmath>
#include <vector>

#include "../data_structures/active_set.h"
#include "../kernels/ahead.h"
#include "../kernels/expand_pull.h"
#include "../kernels/expand_push.h"
#include "../kernels/filter.h"
#include "../kernels/misc.h"
#include "../kernels/pb.h"
#include "../kernels/pull_rows.h"
#include "../kernels/twod.h"
#include "config.h"
#include "features.h"
#include "inspector.h"
#include "statistics.h"

// One record per expand, for logs, training data and roofline accounting.
struct level_record_t {
  int level;
  int dir, fmt, lb, fused, sorted;
  int kernel;              // pulls: 0 length-binned / merge-path, 1 segmented,
                           // 2 propagation blocking or, on a graph it is
                           // slower for, whole rows (pull_kernel in effect)
  bool rows;               // whole rows ran: verts is the number of targets
  long long frontier;      // input frontier length (queue) or n (bitmap)
  long long active, inactive;
  long long edges;         // edges inspected by the expand (device counter)
  long long verts;         // frontier vertices expanded
  float ms;                // expand time (device clock, first to last workgroup)
};

struct executor_t {
  bool profile = true;
  std::vector<level_record_t> log;
  double clock_khz = 0;  // device wall clock

  void clear_log() { log.clear(); }
  void release() { clear_log(); }

  void need_clock() {
    if (clock_khz > 0) return;
    int dev = 0, khz = 0;
    H_ERR(hipGetDevice(&dev));
    H_ERR(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    GSW_REQUIRE(khz > 0, gsw::E_HIP, "device reports no wall clock rate");
    clock_khz = khz;
  }

  // Work counters and times of all logged expands (one report).
  void finalize_log(active_set_t &as) {
    if (log.empty() || !as.dg_work_base) return;
    need_clock();
    const int64_t rows = std::min<int64_t>((int64_t)log.size(), WORK_ROWS);
    const unsigned long long *w = as.read_work(rows);
    for (size_t i = 0; i < log.size(); ++i) {
      const unsigned long long *r = w + std::min<size_t>(i, (size_t)rows - 1) * WORK_N;
      log[i].edges = (long long)r[WORK_EDGES];
      log[i].verts = log[i].rows ? (long long)as.size : (long long)r[WORK_VERTS];
      // (an expand without a workgroup that counted has no stamps)
      if (profile && r[WORK_END] > ~r[WORK_BEGIN])
        log[i].ms = (float)((double)(r[WORK_END] - ~r[WORK_BEGIN]) / clock_khz);
    }
  }

  // ------------------------------------------------------------- filter
  template <typename G, typename F>
  void filter(active_set_t &as, G &g, F &f, stat_t &stat, feature_t &fets,
              config_t &conf) {
    const double s = stat.last_filter_time;
    as.set_fmt(conf.conf_asfmt);
    if (conf.conf_asfmt == Queue) {
      bool tofilter = !conf.conf_fuse_inspect;
      if (conf.conf_switch_to_fusion) {
        tofilter = true;
        conf.conf_switch_to_fusion = false;
      }
      if (conf.conf_first_round) tofilter = true;
      if (tofilter) {
        if (!(as.queue.mode == Cached && as.queue.traceback))
          run_filter(as, conf);
      }
      // a fused level of a non-idempotent algorithm de-duplicates its
      // pushes within the level only: start from a clean `visited`, also on
      // the level that switches into fusion (an earlier fused phase may have
      // left marks behind)
      if (conf.conf_fuse_inspect && !conf.conf_pruning)
        gsw::fill_async<uint64_t>(as.bitmap.visited.dg_bits, 0,
                                  as.bitmap.visited.n_words + 1);
      as.swap_queues();
    }
    conf.thdnum = gsw::BLOCK;
    if (!conf.conf_fuse_inspect) {
      const double wl = (conf.conf_dir == Push) ? fets.push_workload
                                                : fets.pull_workload;
      conf.ctanum = (int)MIN(256.0, wl / conf.thdnum / 2 + 1);
      if (conf.ctanum < 4)
        conf.conf_idle += 1;
      else
        conf.conf_idle = 0;
      if (conf.ctanum < 5 && conf.conf_lb == STRICT && !conf.force.has_lb &&
          !conf.policy_mlp)
        conf.conf_lb = CM;
    }
    if constexpr (std::is_same<G, device_graph_t<CSR, typename G::edge_t>>::value) {
      // fused levels skip the inspector, so the filter's per-vertex update
      // is applied to the queued vertices here (kernel_fusion.cuh:84-96)
      if (conf.conf_compensation && conf.conf_centric == VC &&
          conf.conf_fuse_inspect && !conf.conf_first_round &&
          as.fmt == Queue) {
        hipLaunchKernelGGL((gsw::k_compensation<G, F>),
                           dim3(gsw::grid_for(as.get_size_host())),
                           dim3(gsw::BLOCK), 0, gsw::stream(), as, g, f);
        H_ERR(hipGetLastError());
      }
    }
    const double e = gsw_now_ms();
    stat.level = g.level;
    stat.last_filter_time = e - s;
    stat.avg_filter_time =
        (stat.avg_filter_time * g.level + stat.last_filter_time) / (g.level + 1);
    fets.last_filter_time = stat.last_filter_time;
    fets.avg_filter_time = stat.avg_filter_time;
  }

  void run_filter(active_set_t &as, const config_t &conf) {
    const int64_t n = as.size;
    const int64_t nw = (n + 63) >> 6;
    const Status target = conf.conf_target;
    queue_t &q = as.queue;
    const int out_slot = (q.mode == Normal) ? (q.cursor ^ 1) : (q.cursor + 1);
    int32_t *out = (q.mode == Normal) ? q.buf[q.cursor ^ 1] : q.buf[0] + q.offset_out;
    int32_t *out_size = q.sizes + out_slot;
    const long long expect =
        (target == Active) ? as.known_active
        : (target == Inactive) ? as.known_inactive
                               : as.known_active + as.known_inactive;
    GSW_REQUIRE(expect <= (q.mode == Normal ? q.capacity : q.capacity - q.offset_out),
                gsw::E_OVERFLOW, "frontier does not fit the queue");
    const bool normal = q.mode == Normal;
    if (!normal || !q.slot_zero[out_slot]) gsw::set_one_async<int32_t>(out_size, 0);
    if (normal) q.slot_zero[out_slot] = false;
    if (!conf.conf_sorted) {
      const int wpw = gsw::filter_wpw(nw);
      // (the consumed length is left alone where it is known to be zero)
      int32_t *consumed = normal && !q.slot_zero[q.cursor] ? q.sizes + q.cursor : nullptr;
      hipLaunchKernelGGL(gsw::k_filter_unsorted,
                         dim3(gsw::grid_for((nw + wpw - 1) / wpw, gsw::BLOCK / gsw::WAVE, 1024)),
                         dim3(gsw::BLOCK), 0, gsw::stream(), as, target, n, wpw, out,
                         out_size, consumed);
      q.consumed_clear = consumed != nullptr;
    } else {
      const int nb = (int)MAX(1, MIN(1024, (nw + gsw::BLOCK - 1) / gsw::BLOCK));
      const int64_t wpb = (nw + nb - 1) / nb;
      as.ensure_block_count(nb);
      hipLaunchKernelGGL(gsw::k_filter_sorted_count, dim3(nb), dim3(gsw::BLOCK),
                         0, gsw::stream(), as, target, n, wpb, as.dg_block_count);
      hipLaunchKernelGGL(gsw::k_filter_sorted_write, dim3(nb), dim3(gsw::BLOCK),
                         0, gsw::stream(), as, target, n, wpb, as.dg_block_count,
                         out, out_size);
    }
    H_ERR(hipGetLastError());
    q.host_sizes[out_slot] = (int)expect;
  }

  // ------------------------------------------------------------- expand
  template <typename G, typename F>
  void expand(active_set_t &as, G &g, F &f, stat_t &stat, feature_t &fets,
              config_t &conf) {
    const double s = gsw_now_ms();
    // WM and CM scan the degrees of a wavefront's (64) or a workgroup's
    // (256) frontier vertices in int32; where the graph's degrees could
    // overflow that sum the level runs STRICT (int64 prefixes), forced
    // choices included
    if ((conf.conf_lb == WM || conf.conf_lb == CM) &&
        fets.max_deg * gsw::BLOCK > (double)INT32_MAX)
      conf.conf_lb = STRICT;
    level_record_t rec{};
    rec.level = g.level;
    rec.dir = conf.conf_dir;
    rec.fmt = as.fmt;
    rec.lb = conf.conf_lb;
    rec.fused = conf.conf_fuse_inspect;
    rec.sorted = conf.conf_sorted;
    rec.kernel = conf.conf_dir == Pull ? (!conf.mp_pull ? 1 : conf.pb_pull ? 2 : 0) : 0;
    rec.frontier = as.get_size_host();
    rec.active = as.known_active;
    rec.inactive = as.known_inactive;
    as.select_work_row((int)log.size());
    {
      // WM push: about 128 edges per wavefront at the frontier's mean degree
      // (the last inspected one on fused levels); measured against 64 edges
      // and against filling the capped grid first, this target keeps
      // long-range grids at fixed-64 speed and still halves ER levels
      const double d = fets.cur_avg_deg_active > 0 ? fets.cur_avg_deg_active
                                                   : fets.avg_deg;
      int vpw = gsw::WAVE;
      while (vpw > 8 && vpw * d > 128.0) vpw >>= 1;
      conf.wm_vpw = vpw;
      // early-exit TM pulls probe each target's first in-edge from the
      // per-vertex copy when a random in-edge is likely to end the walk:
      // the frontier holds >= 10% of the edges (on R-MAT, where the first
      // in-neighbour is a hub, far more walks end there)
      conf.pull_first = conf.conf_pruning && fets.push_workload_ratio >= 0.1;
    }
    // (a queue of the active vertices, or of the inactive ones)
    conf.work_hint = 0;
    if (!conf.conf_fuse_inspect && as.fmt == Queue) {
      if (conf.conf_dir == Push && conf.conf_target == Active)
        conf.work_hint = fets.push_workload;
      else if (conf.conf_dir == Pull && conf.conf_target == Inactive)
        conf.work_hint = fets.pull_workload;
    }
    if (conf.conf_fuse_inspect && as.queue.mode == Normal)
      as.queue.slot_zero[as.queue.cursor ^ 1] = false;
    rec.rows = dispatch(as, g, f, conf, stat);
    log.push_back(rec);
    if (conf.verbose) {
      std::printf("level %d frontier %lld ", rec.level, rec.frontier);
      conf.show_hints(std::cout);
      std::cout << std::endl;
    }
    if (conf.conf_fuse_inspect && conf.conf_centric == VC) {
      // the next queue's length: grid size for the next level, convergence
      const int out_slot = (as.queue.mode == Normal) ? (as.queue.cursor ^ 1)
                                                     : (as.queue.cursor + 1);
      const bool learned = conf.policy_mlp && stat.learned();
      int nq = as.read_qsize_device(out_slot);
      as.known_active = nq;
      as.check_overflow_cached();
      if (nq == 0) as.halt_host();
      // Learned selector on fused levels: a small next frontier stays fused
      // with the current class; a large one (where a pull or another format
      // may win) is handed to the next level's inspector, whose fused
      // inference picks the variant.
      if (learned) {
        if (conf.mlp_entered_fused) {  // the inspector chose fused for this level
          conf.mlp_fused_ref = rec.frontier;
          conf.mlp_entered_fused = false;
        }
        if (nq > 0 && (double)nq * gsw_mlp::INSPECT_FRACTION >= (double)as.size &&
            (double)nq >= gsw_mlp::INSPECT_GROWTH * (double)conf.mlp_fused_ref) {
          conf.conf_fuse_inspect = false;
          conf.conf_fusion = false;
          as.swap_queues();
        }
      }
    }
    const double e = gsw_now_ms();
    const int L = g.level > 0 ? g.level : 1;
    stat.last_expand_time = e - s;
    stat.last_time = stat.last_filter_time + stat.last_expand_time;
    stat.avg_time = (stat.avg_time * (L - 1) + stat.last_time) / L;
    stat.avg_expand_time = (stat.avg_expand_time * (L - 1) + stat.last_expand_time) / L;
    fets.last_expand_time = stat.last_expand_time;
    if (fets.pattern == Idem && fets.avg_expand_time > 0 &&
        fets.last_expand_time > 5 * fets.avg_expand_time &&
        conf.conf_fuse_inspect && !conf.force.has_fusion && !conf.policy_mlp) {
      conf.conf_fuse_inspect = false;
      as.swap_queues();
    }
    fets.avg_expand_time = stat.avg_expand_time;
    fets.last_time = stat.last_time;
    fets.avg_time = stat.avg_time;
    conf.conf_first_round = false;
  }

  // After a fused expand whose next queue is not empty: further fused levels
  // without the host (kernels/ahead.h), at most max_levels. Returns how many
  // ran and leaves the state as the last one's expand() would. The rule
  // selector's fused WM push only: the learned selector looks at every fused
  // level's queue length.
  template <typename G, typename F>
  int run_ahead(active_set_t &as, G &g, F &f, feature_t &fets, config_t &conf,
                int64_t max_levels) {
    using namespace gsw;
    if (!conf.conf_fuse_inspect || conf.conf_centric != VC || conf.policy_mlp ||
        conf.verbose || conf.conf_compensation || conf.conf_lb != WM || as.fmt != Queue ||
        as.queue.mode != Normal || as.converged || as.known_active <= 0)
      return 0;
    hipStream_t st = stream();
    need_clock();
    queue_t &q = as.queue;
    const bool prune = conf.conf_pruning;
    if (!as.dg_ahead) H_ERR(hipMalloc(&as.dg_ahead, sizeof(ahead_t)));
    if (!as.h_ahead) {
      H_ERR(hipHostMalloc((void **)&as.h_ahead, sizeof(long long) * (AHEAD_WORDS + 3)));
      as.h_ahead[AHEAD_WORDS + 2] = 0;
    }
    if (!prune && !as.ahead_bits.dg_bits) as.ahead_bits.build(as.size);
    ahead_t *a = (ahead_t *)as.dg_ahead;
    long long *h = as.h_ahead, *mark = h + AHEAD_WORDS + 2;
    const ahead_t *ha = (const ahead_t *)h;
    uint64_t *const bits[2] = {as.bitmap.visited.dg_bits, as.ahead_bits.dg_bits};
    const int64_t n_bits = prune ? 0 : as.bitmap.visited.n_words;
    // the exit rule of expand(): a level's device time, with the host's share
    // that its levels have (about 25 us), against the average of the levels
    // before it, expand()'s included
    const bool rule = fets.pattern == Idem && !conf.force.has_fusion;
    const double share = clock_khz * 0.025;
    double levels = (double)MAX(1, g.level);
    double ticks = fets.avg_expand_time * clock_khz * levels;
    const int per = BLOCK / (WAVE / conf.wm_vpw);  // frontier vertices per workgroup
    const double size = (double)as.size;
    int ran = 0, in_buf = q.cursor ^ 1;  // buffer of the next input
    bool begin = true, slow = false;
    long long nq = as.known_active;
    double growth = (double)nq / (double)MAX(1LL, log.back().frontier);
    while (nq > 0 && !slow) {
      int k = (int)MIN((int64_t)AHEAD, max_levels - ran);
      k = (int)MIN((int64_t)k, (int64_t)WORK_ROWS - 1 - (int64_t)log.size());
      if (k <= 0) break;
      // Grids for twice the growth seen last (four times where it is fast). A
      // level that outgrows its grid is launched again: a second round of a
      // grid's wavefronts costs more (a tree of fan-out 16 from three roots,
      // 4124 vertices: 84 us, 193 on a grid of a third). An explosion (a
      // random graph's) is followed level by level once it reaches a good
      // part of the graph, and from the start where it is so steep that its
      // second level may be one for the exit rule (a tree of fan-out 64: 308
      // us with the rule, 540 when its three levels ran as one batch).
      const double margin = growth > 2 ? 4 : 2;
      int grids[AHEAD];
      double est = (double)nq, reach[AHEAD];
      for (int j = 0; j < k; ++j) {
        const double up = j == 0 ? est : MIN(size, margin * est);
        grids[j] = (int)MAX(1.0, MIN((double)MAX_GRID, std::ceil(up / per)));
        reach[j] = grids[j] >= MAX_GRID ? 2147483647.0 : (double)grids[j] * per;
        est = MIN(size, est * MAX(growth, 1.25));
        if ((growth > 2 && est * 32 > size) || growth > 20) k = j + 1;
      }
      if (begin)
        hipLaunchKernelGGL(k_ahead_begin, dim3(grid_for(ran == 0 ? n_bits : 1)), dim3(BLOCK),
                           0, st, a, ran % AHEAD_SLOTS, (int)nq, bits[0], bits[1],
                           ran == 0 ? n_bits : 0);
      for (int j = 0; j < k; ++j) {
        const int i = ran + j;
        as.select_work_row((int)log.size() + j);
        active_set_t la = as;
        la.queue.cursor = in_buf ^ (j & 1);
        // (output_size() is sizes + (cursor ^ 1): the slot after the input's)
        la.queue.sizes = a->q + (i + 1) % AHEAD_SLOTS - (la.queue.cursor ^ 1);
        if (!prune) la.bitmap.visited.dg_bits = bits[i & 1];
        G gl = g;
        gl.level = g.level + 1 + j;
        using Bd = push_body<G, F, true>;
        hipLaunchKernelGGL(k_push_wm_ahead<Bd>, dim3(grids[j]), dim3(BLOCK), 0, st,
                           Bd{la, gl, f, conf, prune ? nullptr : bits[(i & 1) ^ 1]},
                           conf.wm_vpw, a, j, i % AHEAD_SLOTS, (int)reach[j]);
      }
      const long long seq = *mark + 1;
      hipLaunchKernelGGL(k_ahead_end, dim3(1), dim3(64), 0, st, (const ahead_t *)a,
                         (const int32_t *)as.dg_ctrl, h, mark, seq);
      H_ERR(hipGetLastError());
      await_mark(mark, seq, st);
      GSW_REQUIRE(h[AHEAD_WORDS + 1] == 0, E_OVERFLOW, "frontier queue overflow");
      begin = false;
      level_record_t rec = log.back();
      int done = 0;
      for (int j = 0; j < k; ++j) {
        if (ha->sizes[j] == 0) break;
        if ((double)ha->sizes[j] > reach[j]) {
          begin = true;  // its length back into the slot
          break;
        }
        rec.level = ++g.level;
        rec.frontier = rec.active = ha->sizes[j];
        rec.inactive = as.known_inactive;
        log.push_back(rec);
        ++done;
        const double dt =
            share + (double)((j + 1 < k ? ha->clock[j + 1] : h[AHEAD_WORDS]) - ha->clock[j]);
        if (rule && dt > 5 * (ticks / levels)) slow = true;
        ticks += dt;
        levels += 1;
      }
      nq = done < k ? ha->sizes[done] : ha->q[(ran + k) % AHEAD_SLOTS];
      if (done > 0) growth = (double)nq / (double)log.back().frontier;
      ran += done;
      in_buf ^= done & 1;
    }
    if (ran == 0) return 0;
    // as after expand(): the cursor on the consumed queue, the next one's
    // length behind it
    q.cursor = in_buf ^ 1;
    q.slot_zero[0] = q.slot_zero[1] = false;
    set_one_async<int32_t>(q.sizes + in_buf, (int)nq);
    q.host_sizes[in_buf] = (int)nq;
    as.known_active = nq;
    if (nq == 0) as.halt_host();
    if (slow && nq > 0) {
      conf.conf_fuse_inspect = false;
      as.swap_queues();
    }
    return ran;
  }

  // true where the whole-row pull ran
  template <typename G, typename F>
  bool dispatch(active_set_t &as, G &g, F &f, config_t &conf, stat_t &stat);
};

// grid for a frontier of N items processed `per` items per workgroup
inline int expand_grid(int64_t N, int per) {
  int64_t g = (N + per - 1) / per;
  return (int)MAX(1, MIN((int64_t)gsw::MAX_GRID, g));
}

// slot prefix of a queue frontier of N items into the STRICT workset
template <typename G>
void strict_scan(active_set_t &as, G &g, const config_t &conf, int64_t N, bool pull) {
  using namespace gsw;
  const int64_t nb = (N + SCAN_TILE - 1) / SCAN_TILE;
  if (nb <= SCAN_OWN_TILES) {
    hipLaunchKernelGGL(k_strict_prepare_sums<G>, dim3((unsigned)nb), dim3(BLOCK), 0, stream(),
                       as, g, conf.conf_target, pull, as.workset.dg_scan, as.workset.dg_bsum);
    hipLaunchKernelGGL(k_scan_tile_apply_own, dim3((unsigned)nb), dim3(BLOCK), 0, stream(),
                       as.workset.dg_scan, N, (const int64_t *)as.workset.dg_bsum);
    return;
  }
  hipLaunchKernelGGL(k_strict_prepare<G>, dim3(grid_for(N)), dim3(BLOCK), 0, stream(), as, g,
                     conf.conf_target, pull, as.workset.dg_scan);
  scan_exclusive_inplace(as.workset.dg_scan, N, as.workset.dg_bsum);
}

// STRICT workgroups share the slots evenly: no more of them than 256-slot
// shares where the inspector counted the level's edges (a level of 3 K edges:
// 12 workgroups instead of 2048 that each search for an empty share)
inline int strict_grid(const config_t &conf, int64_t N) {
  if (conf.work_hint <= 0) return gsw::MAX_GRID;
  const double slots = conf.work_hint + (double)N;
  return (int)MAX(1.0, MIN((double)gsw::MAX_GRID, std::ceil(slots / gsw::BLOCK)));
}

template <typename G, typename F>
bool executor_t::dispatch(active_set_t &as, G &g, F &f, config_t &conf,
                          stat_t &stat) {
  using namespace gsw;
  hipStream_t st = stream();
  if constexpr (std::is_same<G, device_graph_t<COO, typename G::edge_t>>::value) {
    const int64_t N = as.get_size_host();
    hipLaunchKernelGGL((k_expand_ec<G, F>), dim3(grid_for(N)), dim3(BLOCK), 0,
                       st, as, g, f);
    H_ERR(hipGetLastError());
    return false;
  } else {
    const int64_t N = as.get_size_host();
    if (N == 0) return false;
    const bool push = conf.conf_dir == Push;
    const bool fused = conf.conf_fuse_inspect;
    LB lb = conf.conf_lb;
    // TWOD serves from-all pulls over a bitmap frontier of an unweighted
    // graph; anything else takes the edge-balanced STRICT path
    bool twod_ok = false;
    if constexpr (!G::has_edata)
      twod_ok = !push && conf.conf_fromall && as.fmt == Bitmap && g.twod;
    if (lb == ELB || (lb == TWOD && !twod_ok)) lb = STRICT;
    using MSG = typename pb_msg<F>::type;
    using WAt = typename F::wa_t;
    const bool use_pb = lb == TWOD && conf.pb_pull && g.pb;
    // every vertex stays active: on graphs that gain by it, whole rows and the
    // filter with them (kernels/pull_rows.h), unless the blocked layout is
    // asked for
    bool use_rows = false;
    if constexpr (pb_has_filter_acc<F>::value && is_ra_pair<F>::value)
      use_rows = use_pb && conf.counts_known && conf.wa_zero &&
                 !std::getenv("GSW_PB_ECAP") && !std::getenv("GSW_PB_GROUPS") &&
                 rows_wanted(*g.rowbins, g.dgr_row_ptr, g.dgr_adj_list, g.nvertexs, g.nedges,
                             (int)sizeof(typename F::ra_t));
    if (use_rows) {
      rows_ensure(*g.rowbins, g.dgr_row_ptr, g.nvertexs);
      if (!f.data.dg_ra2)
        H_ERR(hipMalloc((void **)&f.data.dg_ra2,
                        sizeof(typename F::ra_t) * (g.nvertexs + 1)));
    } else if (use_pb) {
      pb_ensure(g, PB_LDS_BYTES / (int)sizeof(MSG), PB_LDS_BYTES / (int)sizeof(WAt));
      pb_vals(*g.pb, sizeof(MSG));
    } else if (lb == TWOD) {
      // slice width from the bytes of source state one message reads
      constexpr int64_t src_bytes = sizeof(typename F::ra_t) > 4 ? sizeof(typename F::ra_t) : 4;
      twod_ensure(g, src_bytes);
    }
    // Scratch must exist before any kernel body copies `as` by value.
    if (lb == TWC && push) as.bins.ensure(as.size);
    if (lb == STRICT) as.workset.ensure(as.size);
    GSW_REQUIRE(!(lb == TWC && push) || (as.bins.sizes && as.bins.bin[2]),
                E_INTERNAL_CHECK, "TWC bins missing");
    GSW_REQUIRE(lb != STRICT || (as.workset.dg_scan && as.workset.dg_bsum),
                E_INTERNAL_CHECK, "STRICT workset missing");
    if (push) {
      auto launch = [&](auto body) {
        using Bd = decltype(body);
        switch (lb) {
          case TM:
            hipLaunchKernelGGL(k_push_tm<Bd>, dim3(expand_grid(N, BLOCK)),
                               dim3(BLOCK), 0, st, body);
            break;
          case WM:
            hipLaunchKernelGGL(k_push_wm<Bd>,
                               dim3(expand_grid(N * (WAVE / conf.wm_vpw), BLOCK)),
                               dim3(BLOCK), 0, st, body, conf.wm_vpw);
            break;
          case CM:
            hipLaunchKernelGGL(k_push_cm<Bd>, dim3(expand_grid(N, BLOCK)),
                               dim3(BLOCK), 0, st, body);
            break;
          case TWC: {
            fill_async<int32_t>(as.bins.sizes, 0, 4);
            hipLaunchKernelGGL(k_twc_bin<G>, dim3(expand_grid(N, BLOCK)),
                               dim3(BLOCK), 0, st, as, g, conf.conf_target,
                               false, conf.twc_small, conf.twc_large);
            hipLaunchKernelGGL(k_push_twc<Bd>, dim3(expand_grid(N, BLOCK)),
                               dim3(BLOCK), 0, st, body);
            break;
          }
          default: {  // STRICT
            const int64_t *scan = nullptr;  // bitmap: implicit rows[v] + v
            if (as.fmt == Queue) {
              strict_scan(as, g, conf, N, false);
              scan = as.workset.dg_scan;
            }
            hipLaunchKernelGGL(k_push_strict<Bd>, dim3(strict_grid(conf, N)), dim3(BLOCK),
                               0, st, body, scan);
            break;
          }
        }
        H_ERR(hipGetLastError());
      };
      if (fused)
        launch(push_body<G, F, true>{as, g, f, conf});
      else
        launch(push_body<G, F, false>{as, g, f, conf});
    } else {
      using Bd = pull_body<G, F>;
      // (one group only: with several, a later group's phase 1 would read
      // ranks an earlier group's filter had already updated)
      conf.pb_fuse_filter = use_pb && conf.counts_known && g.pb->ng == 1;
      Bd body{as, g, f, conf};
      switch (lb) {
        case TM:
          if constexpr (is_level_sync<F>::value) {
            if (as.fmt == Bitmap && !conf.conf_fromall && !conf.conf_toall) {
              // this level's pull also inspects the next one
              gsw_mlp::sel_dev_t d;
              if (conf.policy_mlp && stat.mlp.w) {
                d = stat.mlp;
                d.level = (float)g.level;
              }
              hipLaunchKernelGGL(k_pull_tm_inspect<Bd>,
                                 dim3(grid_for((g.nvertexs + 63) / 64 * 64)),
                                 dim3(BLOCK), 0, st, body,
                                 as.bitmap.visited.dg_bits, stat.slots());
              hipLaunchKernelGGL(k_stat_finish, dim3(1), dim3(BLOCK), 0, st, d,
                                 stat.slots(), stat.h_runtime_info, ++stat.seq);
              H_ERR(hipGetLastError());
              // the next frontier becomes `active`; the old active words
              // (vertices reached earlier) become the `visited` marks
              std::swap(as.bitmap.active.dg_bits, as.bitmap.visited.dg_bits);
              conf.conf_pre_inspected = true;
              break;
            }
          }
          hipLaunchKernelGGL(k_pull_tm<Bd>, dim3(expand_grid(N, BLOCK)),
                             dim3(BLOCK), 0, st, body);
          break;
        case WM:
        case TWC:
          hipLaunchKernelGGL(k_pull_wm<Bd>, dim3(expand_grid(N, BLOCK)),
                             dim3(BLOCK), 0, st, body);
          break;
        case CM:
          hipLaunchKernelGGL(k_pull_cm<Bd>, dim3(expand_grid(N, BLOCK)),
                             dim3(BLOCK), 0, st, body);
          break;
        case TWOD: {
          if constexpr (pb_has_filter_acc<F>::value && is_ra_pair<F>::value) {
            if (use_rows) {
              const rowbins_t &rb = *g.rowbins;
              int4 first;
              first.x = rows_blocks(rb, 3);
              first.y = first.x + rows_blocks(rb, 2);
              first.z = first.y + rows_blocks(rb, 1);
              first.w = first.z + rows_blocks(rb, 0);
              F out = f;
              std::swap(out.data.dg_ra, out.data.dg_ra2);
              hipLaunchKernelGGL((k_pull_rows<Bd, F>), dim3(first.w), dim3(BLOCK), 0, st,
                                 body, out, rb, first);
              std::swap(f.data.dg_ra, f.data.dg_ra2);
              conf.filter_done = true;
              break;
            }
          }
          if (use_pb) {
            // propagation blocking: messages to slots, then slots to targets
            // group by group (consecutive bins): a group's phase 2 follows
            // its own phase 1
            const pb_t &pb = *g.pb;
            for (int64_t k = 0; k < pb.ng; ++k) {
              pb_t q = pb;
              q.p1 = pb.p1 + 4 * pb.g1h[k];
              q.p2 = pb.p2 + 4 * pb.g2h[k];
              const int64_t n1 = pb.g1h[k + 1] - pb.g1h[k];
              const int64_t n2 = pb.g2h[k + 1] - pb.g2h[k];
              if (n1 > 0)
                hipLaunchKernelGGL((k_pb_scatter<Bd, MSG>), dim3(n1), dim3(PB_BLOCK),
                                   0, st, body, q);
              if (n2 > 0)
                hipLaunchKernelGGL((k_pb_gather<Bd, MSG>), dim3(n2), dim3(PB_BLOCK), 0,
                                   st, body, q);
            }
            if (conf.pb_fuse_filter) {
              // targets of bins split over workgroups: filtered once all
              // parts are added
              if (pb.nsplit > 0)
                hipLaunchKernelGGL((k_pb_filter_split<Bd>),
                                   dim3(grid_for(pb.nsplit)), dim3(BLOCK), 0, st, body,
                                   (const int32_t *)pb.split, pb.nsplit);
              conf.filter_done = true;
            }
            break;
          }
          // the slices one after another (each launch owns its targets)
          const twod_t &tw = *g.twod;
          for (int p = 0; p < tw.P; ++p) {
            const twod_slice_t &sl = tw.s[p];
            if (sl.ne == 0) continue;
            if (conf.mp_pull) {
              int grid = 0;
              for (int c = 0; c <= TWOD_BINS; ++c) grid += sl.blocks[c];
              hipLaunchKernelGGL(k_pull_bins<Bd>, dim3(grid), dim3(BLOCK), 0, st,
                                 body, sl);
            } else {
              const int64_t tiles = (sl.ne + sl.nr + SCHUNK - 1) / SCHUNK;
              const int grid = (int)MIN((int64_t)MAX_GRID, tiles);
              hipLaunchKernelGGL(k_pull_twod<Bd>, dim3(grid), dim3(BLOCK), 0, st,
                                 body, sl);
            }
          }
          break;
        }
        default: {  // STRICT
          const int64_t *scan = nullptr;  // bitmap: implicit rows[v] + v
          if (conf.mp_pull && conf.conf_fromall && !conf.conf_pruning &&
              as.fmt == Bitmap) {
            // every in-edge contributes: the merge-path walk is cheaper
            hipLaunchKernelGGL(k_pull_mp<Bd>, dim3(MAX_GRID), dim3(BLOCK), 0,
                               st, body);
            break;
          }
          if (as.fmt == Queue) {
            strict_scan(as, g, conf, N, true);
            scan = as.workset.dg_scan;
          }
          hipLaunchKernelGGL(k_pull_strict<Bd>, dim3(strict_grid(conf, N)), dim3(BLOCK), 0,
                             st, body, scan);
          break;
        }
      }
      H_ERR(hipGetLastError());
    }
    return use_rows;
  }
}
