// PageRank against the template API, with the optional filter_acc member and
// the flags that let a blocked pull apply it. GSW_APP_ITERS iterations;
// GSW_APP_OUT=<file> gets the read attribute (float per vertex).
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "gswitch.h"

using G = device_graph_t<CSR, Empty>;

inspector_t inspector;
selector_t selector;
executor_t executor;
feature_t fets;
config_t conf;
stat_t stats;

// PageRank with a fixed number of iterations: WA accumulates, RA holds the
// rank per out-degree; filter_acc is the filter given the accumulated value.
struct Rank : Functor<VC, double, float, Empty> {
  double damp;
  __device__ Status filter(int v, G g) {
    const double acc = *wa_of(v);
    *wa_of(v) = 0;
    return filter_acc(v, acc, g);
  }
  __device__ Status filter_acc(int v, double acc, G g) {
    const int od = g.get_out_degree(v);
    const double r = acc * damp + (1 - damp);
    *ra_of(v) = (float)(od ? r / od : r);
    return Active;
  }
  __device__ double emit(int v, Empty *e, G g) { return (double)*ra_of(v); }
  __device__ bool comp(double *v, double msg, G g) {
    *v += msg;
    return true;
  }
  __device__ bool compAtomic(double *v, double msg, G g) {
    atomicAdd(v, msg);
    return true;
  }
};

// The functor by value, as the reference's drivers take it. False if the
// records change when they are read again.
template <typename Gd, typename F> bool iterate(Gd g, F f, int iters) {
  active_set_t as = build_active_set(g.nvertexs, conf);
  as.init();
  for (int level = 0;; ++level) {
    inspector.inspect(as, g, f, stats, fets, conf);
    if (as.finish(g, f, conf) || level == iters) break;
    selector.select(stats, fets, conf);
    executor.filter(as, g, f, stats, fets, conf);
    g.update_level();
    executor.expand(as, g, f, stats, fets, conf);
    if (as.finish(g, f, conf)) break;
  }
  executor.finalize_log(as);
  const std::vector<level_record_t> once = executor.log;
  executor.finalize_log(as);
  bool same = (int)once.size() == iters;
  for (size_t i = 0; i < once.size(); ++i)
    same = same && once[i].edges == g.nedges && executor.log[i].edges == once[i].edges &&
           executor.log[i].ms == once[i].ms;
  return same;
}

int main(int argc, char *argv[]) {
  parse_cmd(argc, argv, "rank");
  fets.centric = VC;
  fets.pattern = ASSO;
  fets.fromall = true;
  fets.toall = true;
  conf.pb_pull = true;
  conf.counts_known = true;
  conf.wa_zero = true;

  auto g = build_graph<VC>(cmd_opt.path, fets, cmd_opt.with_header,
                           cmd_opt.with_weight, cmd_opt.directed);
  if (g.hg.nedges == 0) return 1;
  Rank f;
  f.damp = 0.85;
  f.data.build(g.hg.nvertexs);
  f.data.init_wa([](int) { return 0.0; });
  f.data.init_ra([&](int v) {
    const int64_t od = g.hg.start_pos[v + 1] - g.hg.start_pos[v];
    return (float)((1 - 0.85) / (double)(od ? od : 1));
  });
  init_conf(stats, fets, conf, g, f);
  const char *iters = std::getenv("GSW_APP_ITERS");
  if (!iterate(g.dg, f, iters ? std::atoi(iters) : 10)) return 2;
  f.data.sync_ra();
  if (const char *out = std::getenv("GSW_APP_OUT")) {
    FILE *fp = std::fopen(out, "wb");
    std::fwrite(f.data.h_ra, sizeof(float), g.hg.nvertexs, fp);
    std::fclose(fp);
  }
  return 0;
}
