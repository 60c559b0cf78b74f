"""The work that users of the framework have it do, as measurable cases.

Every case is one query on a device-resident graph through the Python binding
(gswitch_amd.Graph): the graph is uploaded once, as a program that queries it
keeps it, and a pass is one call with its results, in host memory where the
call puts them there. Graphs come in the families of this repository's own
configurations: R-MAT (a = 0.57, b = c = 0.19), 4-neighbour grids with one edge
in ten deleted and one long-range edge per hundred, and batches of independent
random graphs. They are made on the GPU from the seed alone.
"""
import math

import numpy as np
import torch

import gswitch_amd as gsw

DEV = "cuda"


def listed():
    return [
        # the smallest interactive query: launches and host round trips count
        dict(name="bfs_rmat12", op="bfs", graph="rmat", scale=12, degree=16,
             shuffle=False, capture=0),
        # hop distances over a large social graph, one query at a time, by the
        # device-resident direction-optimising loop
        dict(name="bfs_device_rmat22", op="bfs", graph="rmat", scale=22, degree=16,
             shuffle=False, capture=8),
        # hop distances over a road- or mesh-like graph: many levels
        dict(name="bfs_grid1500", op="bfs", graph="grid", rows=1500, cols=1377,
             shuffle=False, capture=0),
        # weighted distances in a social graph whose ids carry no order
        dict(name="sssp_rmat18", op="sssp", graph="rmat", scale=18, degree=16,
             shuffle=True),
        # weighted distances over a road-like graph
        dict(name="sssp_grid1000", op="sssp", graph="grid", rows=1000, cols=1023,
             shuffle=False),
        # components of a large social graph
        dict(name="cc_rmat21", op="cc", graph="rmat", scale=21, degree=16, shuffle=False,
             inplace=False),
        # components of a mesh into the caller's device buffer, as a serving
        # loop or a captured sequence calls it
        dict(name="cc_inplace_grid3000", op="cc", graph="grid", rows=3000, cols=2851,
             shuffle=False, inplace=True),
        # ranks of a middling directed link graph
        dict(name="pagerank_web16", op="pagerank", graph="web", scale=16, degree=12,
             shuffle=True, iters=30),
        # ranks of a large social graph: the largest case
        dict(name="pagerank_rmat22", op="pagerank", graph="rmat", scale=22, degree=16,
             shuffle=False, iters=20),
        # reachability from 64 sources at once
        dict(name="msbfs64_rmat20", op="msbfs64", graph="rmat", scale=20, degree=16,
             shuffle=False, sources=64),
        # levels and components of many small independent graphs
        dict(name="batch_er300", op="batch", graph="er", count=300, nmin=1000,
             nmax=30000, dmin=2.0, dmax=32.0, capture=8),
        # betweenness dependencies from one root: a forward and a backward pass
        dict(name="bc_rmat17", op="bc", graph="rmat", scale=17, degree=16, shuffle=True),
    ]


def draw(rng):
    op = rng.choice(["bfs", "bfs", "sssp", "sssp", "cc", "cc", "pagerank", "pagerank",
                     "msbfs64", "batch", "bc"])
    if op == "batch":
        nmin = rng.randint(100, 2000)
        return dict(op=op, graph="er", count=int(10 ** rng.uniform(0.7, 2.47)), nmin=nmin,
                    nmax=nmin + int(10 ** rng.uniform(2, 4.4)),
                    dmin=round(rng.uniform(1, 6), 2), dmax=round(rng.uniform(8, 32), 2),
                    capture=rng.choice([4, 8]))
    top = {"bfs": 22, "sssp": 19, "cc": 21, "pagerank": 22, "msbfs64": 20, "bc": 17}[op]
    case = dict(op=op)
    if op == "pagerank" and rng.random() < 0.4:
        case.update(graph="web", scale=rng.randint(9, 17), degree=rng.randint(3, 20),
                    shuffle=rng.random() < 0.7)
    elif op in ("msbfs64", "pagerank") or rng.random() < 0.55:
        case.update(graph="rmat", scale=rng.randint(9, top), degree=rng.randint(3, 16),
                    shuffle=rng.random() < 0.4)
    else:
        side = {"bfs": 1430, "sssp": 1000, "cc": 2900, "bc": 400}[op]
        case.update(graph="grid", rows=int(round(math.exp(rng.uniform(math.log(20),
                                                                     math.log(side))))),
                    cols=int(round(math.exp(rng.uniform(math.log(20), math.log(side))))),
                    shuffle=rng.random() < 0.3)
    if op == "bfs":
        case.update(capture=rng.choice([0, 0, 8]))
    if op == "cc":
        case.update(inplace=rng.random() < 0.4)
    if op == "pagerank":
        case.update(iters=rng.randint(5, 20))
    if op == "msbfs64":
        case.update(sources=rng.choice([64, 64, rng.randint(2, 63)]))
    return case


# ------------------------------------------------------------------ graphs
def _generator(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 17)


def _edges(case, gen):
    """(n, src, dst, offsets): one entry per edge sample, int64, on the GPU."""
    if case["graph"] in ("rmat", "web"):
        n = 1 << case["scale"]
        k = case["degree"] << case["scale"]
        u = torch.zeros(k, dtype=torch.int64, device=DEV)
        v = torch.zeros(k, dtype=torch.int64, device=DEV)
        for _ in range(case["scale"]):
            x = torch.rand(k, device=DEV, generator=gen)
            right, both = x >= 0.76, x >= 0.95
            u = 2 * u + right.long()
            v = 2 * v + (((x >= 0.57) & ~right) | both).long()
        return n, u, v, None
    if case["graph"] == "grid":
        r, c = case["rows"], case["cols"]
        n = r * c
        at = torch.arange(n, device=DEV).view(r, c)
        u = torch.cat([at[:, :-1].reshape(-1), at[:-1].reshape(-1)])
        v = torch.cat([at[:, 1:].reshape(-1), at[1:].reshape(-1)])
        keep = torch.rand(u.numel(), device=DEV, generator=gen) >= 0.1
        far = torch.randint(n, (2, int(0.01 * u.numel()) + 1), device=DEV, generator=gen)
        return n, torch.cat([u[keep], far[0]]), torch.cat([v[keep], far[1]]), None
    # er: independent random graphs numbered one after another; their sizes and
    # mean degrees are the case's, their edges the seed's
    cnt = case["count"]
    i = torch.arange(1, cnt + 1, device=DEV, dtype=torch.float64)
    x, y = (i * 0.7548776662466927) % 1, (i * 0.5698402909980532) % 1
    lo, hi = math.log(case["nmin"]), math.log(case["nmax"])
    size = torch.exp(lo + (hi - lo) * x).long().clamp(case["nmin"], case["nmax"])
    deg = case["dmin"] + (case["dmax"] - case["dmin"]) * y
    k = (size * deg / 2).long()
    off = torch.zeros(cnt + 1, dtype=torch.int64, device=DEV)
    off[1:] = size.cumsum(0)
    which = torch.repeat_interleave(torch.arange(cnt, device=DEV), k)
    p = torch.rand(2, which.numel(), device=DEV, generator=gen, dtype=torch.float64)
    ends = off[which] + (p * size[which]).long()
    return int(off[-1]), ends[0], ends[1], off


def _csr(case, seed):
    """The graph of a case: n, row offsets, source and column of every
    directed edge, weights (SSSP), instance offsets (batches), and a
    generator for what else the case draws."""
    gen = _generator(seed)
    n, u, v, off = _edges(case, gen)
    if case.get("shuffle"):
        perm = torch.randperm(n, device=DEV, generator=gen)
        u, v = perm[u], perm[v]
    key = u * n + v
    if case["graph"] != "web":
        key = torch.cat([key, v * n + u])
    del u, v
    key = torch.unique(key)
    src, col = key // n, key % n
    loop = src == col
    if bool(loop.any()):
        src, col = src[~loop], col[~loop]
    row = torch.zeros(n + 1, dtype=torch.int64, device=DEV)
    row[1:] = torch.bincount(src, minlength=n).cumsum(0)
    w = None
    if case["op"] == "sssp":  # 1 .. 64, the same in both directions of an edge
        a, b = torch.minimum(src, col), torch.maximum(src, col)
        h = (a * 1000003 + b * 8191 + int(seed) * 127) & 0x7FFFFFFF
        h = ((h ^ (h >> 15)) * 0x2C1B3C6D) & 0x7FFFFFFF
        w = 1 + ((h ^ (h >> 12)) & 63)
    return dict(n=n, row=row, src=src, col=col, w=w, off=off, gen=gen)


def _queries(case, c):
    """The vertices a case starts from: ends of random edges, so that most lie
    in the large component."""
    if case["op"] not in ("bfs", "sssp", "msbfs64", "bc"):
        return None
    k = case.get("sources", 1)
    m = c["src"].numel()
    if m == 0:
        return np.zeros(k, np.int32)
    at = torch.randint(m, (k,), device=DEV, generator=c["gen"])
    return c["src"][at].to(torch.int32).cpu().numpy()


def prepare(case, seed):
    c = _csr(case, seed)
    state = dict(case=case, roots=_queries(case, c))
    if case["graph"] == "web":
        host = gsw.from_edges(c["n"], c["src"].to(torch.int32).cpu().numpy(),
                              c["col"].to(torch.int32).cpu().numpy(), directed=True)
        state["g"] = gsw.Graph(host)
    else:
        w = None if c["w"] is None else c["w"].to(torch.int32).cpu().numpy().view(np.uint32)
        state["g"] = gsw.Graph(row_ptr=c["row"].cpu().numpy(),
                               col=c["col"].to(torch.int32).cpu().numpy(), w=w)
    if case["op"] == "batch":
        state["off"] = c["off"].cpu().numpy()
    if case.get("inplace"):
        state["labels"] = torch.empty(c["n"], dtype=torch.int32, device=DEV)
    return state


def run(state):
    case, g = state["case"], state["g"]
    op = case["op"]
    if op == "bfs":
        if case["capture"]:
            return g.bfs(int(state["roots"][0]), capture=case["capture"])
        return g.bfs(int(state["roots"][0]))
    if op == "sssp":
        return g.sssp(int(state["roots"][0])).view(np.int32)
    if op == "cc":
        if case["inplace"]:
            g.cc_noalloc(state["labels"].data_ptr(),
                         stream=torch.cuda.current_stream().cuda_stream)
            return state["labels"]
        return g.cc()
    if op == "pagerank":
        return g.pagerank(damping=0.85, iters=case["iters"])
    if op == "msbfs64":
        masks, sums = g.msbfs64(state["roots"])
        return masks.view(np.int64), sums.view(np.int64)
    if op == "batch":
        return g.batch_bfs_cc(state["off"], capture=case["capture"])
    return g.bc(int(state["roots"][0]))


# ------------------------------------------------------- work and tolerance
def _sizes(case):
    """Vertices and directed edges of a case, as its generator gives them on
    average (duplicate samples and self loops left in)."""
    if case["graph"] in ("rmat", "web"):
        n = 1 << case["scale"]
        return n, (1 if case["graph"] == "web" else 2) * case["degree"] * n
    if case["graph"] == "grid":
        n = case["rows"] * case["cols"]
        return n, int(2 * 0.91 * (2 * n - case["rows"] - case["cols"])) + 2
    lo, hi = case["nmin"], case["nmax"]
    mean = (hi - lo) / math.log(hi / lo) if hi > lo else lo
    n = case["count"] * mean
    return n, n * 0.5 * (case["dmin"] + case["dmax"])


def work(case):
    n, m = _sizes(case)
    graph = 8.0 * n + 4.0 * m  # row offsets and columns, once
    op = case["op"]
    if op == "bfs":
        return dict(bytes=graph + 4 * n)
    if op == "sssp":
        return dict(bytes=graph + 4 * m + 4 * n)
    if op == "cc":
        return dict(bytes=graph + 4 * n)
    if op == "pagerank":  # per iteration: the graph, and every rank read and written
        return dict(bytes=case["iters"] * (graph + 8 * n), flops=case["iters"] * (m + 3 * n))
    if op == "msbfs64":
        return dict(bytes=graph + 8 * n)
    if op == "batch":
        return dict(bytes=graph + 8 * n)
    # bc: the graph once forwards and once backwards, level, paths, dependency
    return dict(bytes=2 * graph + 20 * n, flops=3 * m)


def tolerance(case):
    if case["op"] == "pagerank":
        # ranks are stored in 32 bits between iterations and sums are kept in
        # 64: sums in another order move a rank by one rounding now and then
        return dict(rel=2e-7, max=2e-6)
    if case["op"] == "bc":
        return dict(rel=2e-14)  # 64-bit sums in another order
    return "exact"


# ----------------------------------------------------------- plain 64 bits
def _levels(c, roots):
    lv = torch.full((c["n"],), -1, dtype=torch.int32, device=DEV)
    lv[roots] = 0
    level = 0
    while True:
        hit = c["col"][lv[c["src"]] == level]
        hit = hit[lv[hit] < 0]
        if hit.numel() == 0:
            return lv
        level += 1
        lv[hit] = level


def _components(c):
    lab = torch.arange(c["n"], device=DEV)
    while True:
        new = lab.scatter_reduce(0, c["col"], lab[c["src"]], "amin")
        new = torch.minimum(new, new[new])
        if torch.equal(new, lab):
            return lab.to(torch.int32)
        lab = new


def _distances(c, root):
    far = (1 << 32) - 1
    d = torch.full((c["n"],), far, dtype=torch.int64, device=DEV)
    d[root] = 0
    while True:
        step = (d[c["src"]] + c["w"]).clamp(max=far)
        new = d.scatter_reduce(0, c["col"], step, "amin")
        if torch.equal(new, d):
            return d.cpu().numpy().astype(np.uint32).view(np.int32)
        d = new


def _ranks(c, damping, iters):
    out = torch.bincount(c["src"], minlength=c["n"]).double()
    share = out.clamp(min=1)
    rank = torch.full((c["n"],), 1 - damping, dtype=torch.float64, device=DEV)
    for _ in range(iters):
        acc = torch.zeros_like(rank)
        acc.index_add_(0, c["col"], (rank / share)[c["src"]])
        rank = damping * acc + (1 - damping)
    return rank


def _betweenness(c, root):
    lv = _levels(c, torch.tensor([root], device=DEV))
    paths = torch.zeros(c["n"], dtype=torch.float64, device=DEV)
    paths[root] = 1
    dep = torch.zeros_like(paths)
    tree = (lv[c["src"]] >= 0) & (lv[c["col"]] == lv[c["src"]] + 1)
    src, col = c["src"][tree], c["col"][tree]
    deep = int(lv.max())
    for level in range(deep):
        e = lv[src] == level
        paths.index_add_(0, col[e], paths[src[e]])
    for level in range(deep - 1, -1, -1):
        e = lv[src] == level
        got = torch.zeros_like(dep).index_add_(0, src[e],
                                               (1 + dep[col[e]]) / paths[col[e]])
        dep += got * paths
    return lv, paths, dep


def exact(case, seed):
    c = _csr(case, seed)
    roots = _queries(case, c)
    op = case["op"]
    if op == "bfs":
        return _levels(c, torch.as_tensor(roots[:1], device=DEV).long()).cpu().numpy()
    if op == "sssp":
        return _distances(c, int(roots[0]))
    if op == "cc":
        return _components(c)
    if op == "pagerank":
        return _ranks(c, float(np.float32(0.85)), case["iters"])
    if op == "msbfs64":
        masks = torch.zeros(c["n"], dtype=torch.int64, device=DEV)
        sums = np.zeros(64, np.int64)
        for s, r in enumerate(roots):
            lv = _levels(c, torch.tensor([int(r)], device=DEV))
            bit = (1 << s) - (1 << 64 if s == 63 else 0)
            masks |= torch.where(lv >= 0, bit, 0)
            sums[s] = int(lv.clamp(min=0).sum())
        return masks.cpu().numpy(), sums
    if op == "batch":
        first = c["off"][:-1][c["off"][1:] > c["off"][:-1]]
        return _levels(c, first), _components(c)
    return _betweenness(c, int(roots[0]))
