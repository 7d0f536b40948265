"""Performance cases: the maximum-flow calls a program makes through the package's entry points.

A case is a dict of plain values:

  entry    solve     Context.solve: one call on a host graph (upload, solve, release)
           noalloc   Context.solve_noalloc: the same without device allocations
           rcsr      Context.rcsr_push_relabel: the reference-shaped call on RCSR host arrays
           resident  DeviceGraph.solve and read_cut on an uploaded graph: the minimum cut too
           batch     Context.batch_solve over k graphs
           serve     Server: k requests submitted at once, served until all have completed
  net      rlg       Washington random level graph: b levels of a vertices, capacities 1..10000
           genrmf    b frames of a x a vertices, frame-to-frame capacities 1..10000
           rmat      R-MAT of 2^a vertices, edge factor b, capacities 1..1000, from the vertex of
                     largest out-degree to the one of largest in-degree
           bipartite matching network of a left and b right vertices, about 8 arcs per left
                     vertex, unit capacities
           mix       rlg, genrmf and bipartite networks with a..b vertices (log-uniform)
           matching  bipartite networks, both sides log-uniform in a..b
  algo     tc or vc; layout rcsr, bcsr or bcsr2 (where the entry takes one)
  options  default, or the name of one of the option sets a tuned program keeps (OPTIONS)

Every output is a whole number: flow values, and the sink side of the minimum cut, which is the
same for every maximum preflow (the vertices that can reach the sink in its residual graph).  A
flow assignment is not unique, so none is returned.
"""
import math
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import torch

import wbpr_amd as mf
from wbpr_amd import workloads

OPTIONS = {
    "default": {},
    "rmat": {"cycles_per_relabel": 12, "bfs_block_frontier": 1024, "relabel_time_ratio": 2.0,
             "class_lanes": [4, 8, 16, 64, 256], "forward_hops": -1, "cycle_graphs": 1},
    "genrmf": {"cycles_per_relabel": 674, "bfs_block_frontier": 256, "relabel_time_ratio": 4.0,
               "class_lanes": [4, 4, 8, 16, 256], "forward_hops": 2, "bfs_cooperative": 1},
    "batch_vc": {"batch_algo": 1},
}
SERVER_BYTES = 8 << 30


def listed():
    return [
        # a command-line sized problem solved once: what one call costs, whatever the graph
        {"name": "solve_rlg8", "entry": "solve", "net": "rlg", "a": 8, "b": 8, "algo": "tc",
         "layout": "rcsr", "options": "default"},
        # a small problem inside a loop that must not allocate device memory
        {"name": "noalloc_genrmf9x13", "entry": "noalloc", "net": "genrmf", "a": 9, "b": 13,
         "algo": "vc", "layout": "bcsr", "options": "default"},
        # the reference's own call, on its RCSR arrays
        {"name": "rcsr_genrmf16", "entry": "rcsr", "net": "genrmf", "a": 16, "b": 16,
         "algo": "vc", "layout": "rcsr", "options": "default"},
        # a power-law graph of ordinary size solved once
        {"name": "solve_rmat15", "entry": "solve", "net": "rmat", "a": 15, "b": 16, "algo": "vc",
         "layout": "bcsr2", "options": "default"},
        # the 64 x 64 random level graph, thread-centric, kept on the device
        {"name": "resident_rlg64", "entry": "resident", "net": "rlg", "a": 64, "b": 64,
         "algo": "tc", "layout": "bcsr", "options": "default"},
        # a long ragged grid on the reference's layout and thread-centric algorithm
        {"name": "resident_genrmf29x47", "entry": "resident", "net": "genrmf", "a": 29, "b": 47,
         "algo": "tc", "layout": "rcsr", "options": "default"},
        # the 64 x 64 x 64 Genrmf network with its tuned options: long paths
        {"name": "resident_genrmf64", "entry": "resident", "net": "genrmf", "a": 64, "b": 64,
         "algo": "vc", "layout": "bcsr", "options": "genrmf"},
        # one large matching with library defaults
        {"name": "resident_matching", "entry": "resident", "net": "bipartite", "a": 40009,
         "b": 39019, "algo": "vc", "layout": "bcsr", "options": "default"},
        # the scale-22 R-MAT graph with its tuned options: hubs and bandwidth
        {"name": "resident_rmat22", "entry": "resident", "net": "rmat", "a": 22, "b": 16,
         "algo": "vc", "layout": "bcsr", "options": "rmat"},
        # some dozens of mid-size networks of all kinds in one call
        {"name": "batch_mix96", "entry": "batch", "net": "mix", "k": 96, "a": 1000, "b": 20000,
         "options": "batch_vc"},
        # the 4096-instance matching batch
        {"name": "batch_matching4096", "entry": "batch", "net": "matching", "k": 4096, "a": 256,
         "b": 65536, "options": "default"},
        # a burst of requests on a server that is kept running
        {"name": "serve_mix128", "entry": "serve", "net": "mix", "k": 128, "a": 1000, "b": 50000,
         "options": "default"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    entry = rng.choice(["solve", "noalloc", "rcsr", "resident", "resident", "resident", "batch",
                        "serve"])
    if entry == "batch":
        if rng.random() < 0.5:
            return {"entry": entry, "net": "matching", "k": _log(rng, 16, 1024), "a": 256,
                    "b": _log(rng, 4096, 65536), "options": rng.choice(["default", "batch_vc"])}
        return {"entry": entry, "net": "mix", "k": _log(rng, 16, 256), "a": 1000,
                "b": _log(rng, 4000, 20000), "options": rng.choice(["default", "batch_vc"])}
    if entry == "serve":
        return {"entry": entry, "net": "mix", "k": _log(rng, 16, 256), "a": 1000,
                "b": _log(rng, 4000, 50000), "options": "default"}
    net = rng.choice(["rlg", "genrmf", "rmat", "bipartite"])
    case = {"entry": entry, "net": net, "algo": rng.choice(["tc", "vc"]), "options": "default",
            "layout": {"rcsr": "rcsr", "noalloc": "bcsr"}.get(entry) or rng.choice(
                ["rcsr", "bcsr", "bcsr2"])}
    most = 1 if entry == "resident" else 0  # whole calls on smaller graphs, resident on all sizes
    if net == "rlg":
        case["a"], case["b"] = _log(rng, 6, (64, 256)[most]), _log(rng, 6, (64, 256)[most])
    elif net == "genrmf":
        case["a"], case["b"] = _log(rng, 4, (16, 48)[most]), _log(rng, 4, (24, 56)[most])
        if case["algo"] == "vc" and rng.random() < 0.5:
            case["options"] = "genrmf"
    elif net == "rmat":
        case["a"], case["b"] = rng.randint(9, (14, 20)[most]), rng.randint(4, 16)
        case["algo"] = "vc"  # hubs: one lane per vertex is not used on power-law graphs
        if rng.random() < 0.5:
            case["options"] = "rmat"
    else:
        # sides of about one size: the matchings that are not decided by the smaller side alone
        case["a"] = _log(rng, 4000, (20000, 65536)[most])
        case["b"] = int(case["a"] * rng.uniform(0.96, 1.04))
    return case


def _rmat(scale, factor, seed):
    """R-MAT quadrant recursion (0.57, 0.19, 0.19, 0.05) on the GPU, loops and duplicates dropped."""
    gen = torch.Generator("cuda").manual_seed(seed)
    n, e = 1 << scale, factor << scale
    u = torch.zeros(e, dtype=torch.int64, device="cuda")
    v = torch.zeros_like(u)
    for _ in range(scale):
        r = torch.rand(e, device="cuda", generator=gen)
        u = 2 * u + (r >= 0.76)
        v = 2 * v + (((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
    key = torch.unique((u * n + v)[u != v])  # sorted by tail, then head
    u, v = key // n, key % n
    out = torch.bincount(u, minlength=n)
    into = torch.bincount(v, minlength=n)
    s = int(out.argmax())
    into[s] = -1
    t = int(into.argmax())
    offsets = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    offsets[1:] = torch.cumsum(out, 0)
    cap = torch.randint(1, 1001, (key.numel(),), dtype=torch.int32, device="cuda", generator=gen)
    return mf.Graph(n, offsets.int().cpu().numpy(), v.int().cpu().numpy(), cap.cpu().numpy(), s, t)


def _network(net, a, b, seed):
    seed = workloads.splitmix(seed)
    if net == "rlg":
        return mf.gen_washington_rlg(a, b, 10000, seed)
    if net == "genrmf":
        return mf.gen_genrmf(a, b, 1, 10000, seed)
    if net == "rmat":
        return _rmat(a, b, seed >> 1)
    return mf.gen_bipartite(a, b, 8.0, seed)


def _networks(case, seed):
    """The k graphs of a batch or a burst."""
    if case["net"] == "mix":
        return workloads.serving_requests(mf, case["k"], seed, case["a"], case["b"])[0]
    sizes = workloads.batched_sizes(case["k"], seed, case["a"], case["b"])
    with ThreadPoolExecutor(16) as pool:
        return list(pool.map(lambda i: _network("bipartite", *sizes[i], seed * 1000003 + i),
                             range(case["k"])))


_context = []


def _ctx():
    if not _context:
        _context.append(mf.Context(0))
    return _context[0]


def prepare(case, seed):
    ctx = _ctx()
    entry = case["entry"]
    state = {"case": case, "ctx": ctx, "options": OPTIONS[case["options"]]}
    if entry in ("batch", "serve"):
        state["graphs"] = _networks(case, seed)
        if entry == "serve":
            state["server"] = mf.Server(ctx, SERVER_BYTES, 4)
        return state
    state["algo"] = mf.ALGOS[case["algo"]]
    state["layout"] = mf.LAYOUTS[case["layout"]]
    g = state["graph"] = _network(case["net"], case["a"], case["b"], seed)
    if entry == "resident":
        state["device"] = ctx.upload(g, state["layout"])
    elif entry == "rcsr":
        state["reverse"] = mf.build_layout(g, mf.LAYOUT_RCSR)
        state["out"] = {k: np.zeros(max(size, 1), np.int32) for k, size in
                        (("height", g.n), ("excess", g.n), ("fflows", g.m), ("bflows", g.m))}
    return state


def run(state):
    case, ctx, opts = state["case"], state["ctx"], state["options"]
    entry = case["entry"]
    if entry == "resident":
        res = state["device"].solve(state["algo"], **opts)
        return {"value": res.value, "sink_side": state["device"].read_cut()}
    if entry == "solve":
        return ctx.solve(state["graph"], state["algo"], state["layout"], **opts).value
    if entry == "noalloc":
        return ctx.solve_noalloc(state["graph"], state["algo"], **opts).value
    if entry == "rcsr":
        g, rev, out = state["graph"], state["reverse"], state["out"]
        value, _ = ctx.rcsr_push_relabel(
            state["algo"], g.n, g.m, g.s, g.t, out["height"], out["excess"], g.offsets, g.dst,
            g.cap, out["fflows"], out["bflows"], rev["roffsets"], rev["rdst"], rev["flow_index"],
            **opts)
        return {"value": value, "sink_side": out["height"] < g.n}
    if entry == "batch":
        return ctx.batch_solve(state["graphs"], **opts)[0]
    server = state["server"]
    ids = [server.submit(g) for g in state["graphs"]]
    left = set(ids)
    while left:
        server.progress(wait=True)
        left.difference_update(server.completed())
    return np.array([server.result(i)[0] for i in ids])


def _size(net, a, b):
    """(vertices, arcs) of a network, expected where they are drawn."""
    if net == "rlg":
        return a * b + 2, 3 * a * (b - 1) + 2 * a
    if net == "genrmf":
        return a * a * b, 4 * a * (a - 1) * b + a * a * (b - 1)
    if net == "rmat":
        return 1 << a, 0.95 * (b << a)
    return a + b + 2, a + b + a * min(8, b)


def work(case):
    """Bytes of the CSR arrays read once and the results written once."""
    net, a, b = case["net"], case["a"], case["b"]
    k = case.get("k", 1)
    if net in ("mix", "matching"):
        mean = (b - a) / math.log(b / a)  # of a log-uniform size
        if net == "matching":
            n, m = 2 * mean + 2, 10 * mean
        else:
            n, m = mean, 4.2 * mean
    else:
        n, m = _size(net, a, b)
    out = n + 8 if case["entry"] in ("resident", "rcsr") else 8
    return {"bytes": float(k * (4 * (n + 1) + 8 * m + out)), "flops": 0.0}
