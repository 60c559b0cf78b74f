// A pruning, level-synchronous functor whose update may not run twice: it
// counts how often compAtomic ran for every vertex. Written against the
// template API in the shape of the other applications; GSW_APP_OUT=<file> gets
// the root, then a level and a count per vertex (int32).
#include <cstdio>
#include <cstdlib>

#include "gswitch.h"

using G = device_graph_t<CSR, Empty>;

inspector_t inspector;
selector_t selector;
executor_t executor;
feature_t fets;
config_t conf;
stat_t stats;

struct visit_t {
  int level;
  int hits;  // how often compAtomic ran for the vertex
};

struct Visits : Functor<VC, visit_t, Empty, Empty> {
  static constexpr bool level_sync = true;
  __device__ Status filter(int v, G g) {
    const int l = wa_of(v)->level;
    if (l == g.get_level()) return Active;
    return l < 0 ? Inactive : Fixed;
  }
  __device__ visit_t emit(int v, Empty *e, G g) { return {g.get_level(), 1}; }
  __device__ bool cond(int v, visit_t msg, G g) { return wa_of(v)->level < 0; }
  __device__ bool comp(visit_t *d, visit_t msg, G g) {
    d->level = msg.level;
    d->hits += msg.hits;
    return true;
  }
  __device__ bool compAtomic(visit_t *d, visit_t msg, G g) {
    d->level = msg.level;
    atomicAdd(&d->hits, msg.hits);
    return true;
  }
};

template <typename Gd, typename F> double traverse(Gd g, F f, int root) {
  active_set_t as = build_active_set(g.nvertexs, conf);
  as.init(root);
  const double t0 = mwtime();
  for (int level = 0;; ++level) {
    inspector.inspect(as, g, f, stats, fets, conf);
    if (as.finish(g, f, conf)) break;
    selector.select(stats, fets, conf);
    executor.filter(as, g, f, stats, fets, conf);
    g.update_level();
    executor.expand(as, g, f, stats, fets, conf);
    if (as.finish(g, f, conf)) break;
  }
  return mwtime() - t0;
}

int main(int argc, char *argv[]) {
  parse_cmd(argc, argv, "visits");
  fets.centric = VC;
  fets.pattern = Idem;
  fets.fromall = false;
  fets.toall = false;
  conf.conf_pruning = true;

  auto g = build_graph<VC>(cmd_opt.path, fets, cmd_opt.with_header,
                           cmd_opt.with_weight, cmd_opt.directed);
  if (g.hg.nedges == 0) return 1;
  Visits f;
  f.data.build(g.hg.nvertexs);
  int root = cmd_opt.src;
  if (root < 0) root = g.hg.random_root();
  LOG(" -- root %d\n", root);
  fets.use_root = root;
  f.data.init_wa([root](int i) { return visit_t{i == root ? 0 : -1, 0}; });
  init_conf(stats, fets, conf, g, f);

  const double ms = traverse(g.dg, f, root);
  f.data.sync_wa();
  if (const char *out = std::getenv("GSW_APP_OUT")) {
    FILE *fp = std::fopen(out, "wb");
    std::fwrite(&root, sizeof(int), 1, fp);
    std::fwrite(f.data.h_wa, sizeof(visit_t), g.hg.nvertexs, fp);
    std::fclose(fp);
  }
  std::printf("%.3f\n", ms);
  return 0;
}
