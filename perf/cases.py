"""Performance cases of the SCAN framework: what a user's program has it do,
over the range of sizes, graphs and options it is used with.

Graphs are R-MAT (quadrants .57/.19/.19/.05, any vertex count, an exact
number of edges) and planted
partitions with hubs, as in the repository's configurations and tests; an
R-MAT graph may also have its vertex ids shuffled, as ids of crawled or
hashed inputs are.  All outputs are whole numbers (labels, core flags,
similarity flags, role counts), so there are no 64-bit values to compare with.

Kinds of case:
  scan     one pass over a resident graph, results to host arrays
  flags    the same, with the similarity flag of every entry
  device   one pass whose results stay in device buffers of the caller
  noalloc  the same without device allocation, with the flags
  oneshot  a host graph: upload, one pass, release
  admit    a host graph: admission into a serving engine, one query, removal
  serve    a burst of queries on the graphs of a serving engine
  ooc      one out-of-core pass over a host graph within a device budget
"""
import math

import numpy as np
import torch

import efficientstructuralgraphclusteringongpus_amd as sgc

COUNTS = ("u_edges", "similar_edges", "cores", "clusters", "borders", "hubs", "outliers")
EPS_GRID = [k / 20.0 for k in range(2, 19)]  # 0.10, 0.15, ..., 0.90


def listed():
    return [
        # the smallest call: a few hundred vertices, launches and synchronisation
        {"name": "scan-rmat10", "kind": "scan", "graph": "rmat", "n": 1024, "edges": 6000, "shuffled": False,
         "eps": 0.5, "mu": 5},
        # a caller that may not allocate, all three outputs in its own buffers
        {"name": "noalloc-rmat14", "kind": "noalloc", "graph": "rmat", "n": 16384, "edges": 210000,
         "shuffled": False, "eps": 0.4, "mu": 3},
        # the CPU-runnable configuration of the benchmark
        {"name": "scan-rmat16", "kind": "scan", "graph": "rmat", "n": 65536, "edges": 910000, "shuffled": False,
         "eps": 0.5, "mu": 5},
        # an odd number of vertices, low eps, the per-entry flags wanted too
        {"name": "flags-rmat20", "kind": "flags", "graph": "rmat", "n": 1000003, "edges": 15500001,
         "shuffled": False, "eps": 0.2, "mu": 5},
        # ids in no order, several 2^20-id windows, high eps
        {"name": "scan-rmat22-shuffled", "kind": "scan", "graph": "rmat", "n": 4194304, "edges": 48500000,
         "shuffled": True, "eps": 0.6, "mu": 2},
        # the headline workload at its heaviest eps, results left on the device
        {"name": "device-rmat24", "kind": "device", "graph": "rmat", "n": 16777216, "edges": 260000000,
         "shuffled": False, "eps": 0.2, "mu": 5},
        # communities below a few hubs: cores, borders, hubs and outliers
        {"name": "scan-planted-hubs", "kind": "scan", "graph": "planted", "n": 200000, "community": 100,
         "p_in": 0.5, "inter": 8, "hubs": 16, "eps": 0.2, "mu": 4},
        # tight communities: most edges similar, every later phase at work
        {"name": "scan-planted-tight", "kind": "scan", "graph": "planted", "n": 299993, "community": 50,
         "p_in": 0.8, "inter": 3, "hubs": 0, "eps": 0.35, "mu": 5},
        # the whole run from a host graph to labels
        {"name": "oneshot-rmat20", "kind": "oneshot", "graph": "rmat", "n": 1048576, "edges": 15700000,
         "shuffled": False, "eps": 0.4, "mu": 5},
        # a graph enters a serving engine, is asked once and leaves
        {"name": "admit-rmat18", "kind": "admit", "graph": "rmat", "n": 262144, "edges": 3800000, "shuffled": False,
         "eps": 0.3, "mu": 4},
        # many users at once: a burst of mixed queries over graphs of many sizes
        {"name": "serve-burst", "kind": "serve", "graph": "rmat", "n": 1048576, "edges": 15700000, "graphs": 8,
         "queries": 96, "shuffled": False},
        # a graph larger than the device memory it is given
        {"name": "ooc-rmat20", "kind": "ooc", "graph": "rmat", "n": 1048576, "edges": 15700000, "shuffled": False,
         "bytes_per_entry": 12, "eps": 0.3, "mu": 5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["scan", "scan", "scan", "flags", "device", "device", "noalloc", "oneshot", "admit", "serve", "ooc"])
    case = {"kind": kind, "eps": rng.choice(EPS_GRID[2:]), "mu": rng.randint(2, 20)}
    if kind in ("scan", "device") and rng.random() < 0.45:
        case.update(graph="planted", n=_log_int(rng, 5000, 400000), community=_log_int(rng, 30, 300),
                    p_in=round(rng.uniform(0.05, 0.9), 2), inter=rng.randint(2, 10), hubs=rng.choice([0, 4, 16, 64]))
        return case
    most = {"scan": 6000000, "flags": 3000000, "device": 8000000, "noalloc": 30000, "oneshot": 2500000,
            "admit": 600000, "serve": 1200000, "ooc": 1500000}[kind]
    least = {"oneshot": 4000, "admit": 4000, "serve": 20000, "ooc": 60000}.get(kind, 900)
    n = _log_int(rng, least, most)
    case.update(graph="rmat", n=n, edges=int(n * rng.uniform(5.0, 15.5)), shuffled=rng.random() < 0.3)
    if kind == "serve":
        case.update(graphs=rng.randint(2, 10), queries=rng.randint(8, 128))
        del case["eps"], case["mu"]
    if kind == "ooc":
        case.update(bytes_per_entry=rng.randint(9, 18), eps=rng.choice(EPS_GRID[2:]))
    return case


def _rmat_edges(n, draws, gen):
    """Distinct undirected edges u < v as u * n + v, ascending, from R-MAT draws."""
    u = torch.zeros(draws, dtype=torch.int64, device="cuda")
    v = torch.zeros(draws, dtype=torch.int64, device="cuda")
    scale = max(1, (n - 1).bit_length())
    for _ in range(scale):
        r = torch.rand(draws, generator=gen, device="cuda")
        u.mul_(2).add_(r >= 0.76)
        v.mul_(2).add_(((r >= 0.57) & (r < 0.76)) | (r >= 0.95))
        del r
    if n < 1 << scale:
        u.remainder_(n)
        v.remainder_(n)
    keys = torch.minimum(u, v) * n + torch.maximum(u, v)
    keys = torch.sort(keys[u != v])[0]
    first = torch.ones(keys.numel(), dtype=torch.bool, device="cuda")
    first[1:] = keys[1:] != keys[:-1]
    return keys[first]


def _rmat(n, edges, shuffled, seed):
    """A symmetric R-MAT graph of n vertices and exactly `edges` edges."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    draws = int(1.05 * edges) + 64
    keys = _rmat_edges(n, draws, gen)
    while keys.numel() < edges:
        draws = int(1.3 * draws)
        keys = _rmat_edges(n, draws, gen)
    keys = keys[torch.randperm(keys.numel(), generator=gen, device="cuda")[:edges]]
    u, v = keys // n, keys % n
    if shuffled:
        perm = torch.randperm(n, generator=gen, device="cuda")
        u, v = perm[u], perm[v]
        del perm
    keys = torch.sort(torch.cat([u * n + v, v * n + u]))[0]
    del u, v
    row_ptr = torch.searchsorted(keys, torch.arange(n + 1, dtype=torch.int64, device="cuda") * n)
    adj = (keys % n).to(torch.int32).cpu().numpy()
    row_ptr = row_ptr.cpu().numpy().astype(np.uint64)
    del keys
    torch.cuda.empty_cache()
    return sgc.HostGraph.from_csr(row_ptr, adj, check_symmetry=False)


def _host_graph(case, seed):
    if case["graph"] == "planted":
        return sgc.HostGraph.planted(n=case["n"], communities=max(1, case["n"] // case["community"]),
                                     p_in=case["p_in"], inter_per_vertex=case["inter"], hubs=case["hubs"],
                                     hub_fraction=0.05, seed=seed)
    return _rmat(case["n"], case["edges"], case["shuffled"], seed)


def _serving_state(case, seed):
    rng = np.random.default_rng(seed)
    ctx = sgc.Context(0)
    graphs = [_rmat(max(1000, case["n"] >> i), max(6000, case["edges"] >> i), case["shuffled"], seed + i)
              for i in range(case["graphs"])]
    need = sum(sgc.Server.graph_bytes(g) for g in graphs)
    server = sgc.Server(ctx, need + (64 << 20))
    ids = [(server.add_graph(g)[0], g.n) for g in graphs]
    for g in graphs:
        g.close()
    server.set_batching(9_900_000)
    # as many on each graph, in random order
    asked = rng.permutation(np.arange(case["queries"]) % len(ids))
    queries = [(*ids[int(i)], EPS_GRID[int(rng.integers(len(EPS_GRID)))], int(rng.integers(2, 21))) for i in asked]
    return {"case": case, "ctx": ctx, "server": server, "queries": queries}


def prepare(case, seed):
    if case["kind"] == "serve":
        return _serving_state(case, seed)
    graph = _host_graph(case, seed)
    state = {"case": case, "ctx": sgc.Context(0), "n": graph.n, "m": graph.m}
    if case["kind"] in ("oneshot", "admit", "ooc"):
        state["graph"] = graph
        if case["kind"] == "admit":
            state["server"] = sgc.Server(state["ctx"], sgc.Server.graph_bytes(graph) + (1 << 20))
        if case["kind"] == "ooc":
            state["budget"] = max(sgc.ooc_min_budget(graph, case["eps"]),
                                  48 * graph.n + case["bytes_per_entry"] * graph.m)
        return state
    state["dgraph"] = sgc.DeviceGraph(state["ctx"], graph)
    graph.close()
    if case["kind"] in ("device", "noalloc"):
        state["labels"] = torch.empty(state["n"], dtype=torch.int32, device="cuda")
        state["core"] = torch.empty(state["n"], dtype=torch.uint8, device="cuda")
        if case["kind"] == "noalloc":
            state["sim"] = torch.empty(state["m"], dtype=torch.uint8, device="cuda")
        torch.cuda.synchronize()  # the buffers are the library's from here on
    return state


def _counts(stats):
    return {name: int(getattr(stats, name)) for name in COUNTS}


def _result(result):
    out = {"labels": result.labels, "core": result.core, "counts": _counts(result.stats)}
    if result.sim is not None:
        out["sim"] = result.sim
    return out


def run(state):
    case, ctx = state["case"], state["ctx"]
    kind = case["kind"]
    if kind in ("scan", "flags"):
        return _result(sgc.scan(ctx, state["dgraph"], case["eps"], case["mu"], want_sim=kind == "flags"))
    if kind == "device":
        stats = sgc.scan_device(ctx, state["dgraph"], case["eps"], case["mu"], state["labels"].data_ptr(),
                                state["core"].data_ptr())
        return {"labels": state["labels"], "core": state["core"], "counts": _counts(stats)}
    if kind == "noalloc":
        stats = sgc.scan_device_noalloc(ctx, state["dgraph"], case["eps"], case["mu"], state["labels"].data_ptr(),
                                        state["core"].data_ptr(), state["sim"].data_ptr())
        return {"labels": state["labels"], "core": state["core"], "sim": state["sim"], "counts": _counts(stats)}
    if kind == "oneshot":
        dgraph = sgc.DeviceGraph(ctx, state["graph"])
        try:
            return _result(sgc.scan(ctx, dgraph, case["eps"], case["mu"]))
        finally:
            dgraph.close()
    if kind == "ooc":
        return _result(sgc.scan_ooc(ctx, state["graph"], case["eps"], case["mu"], state["budget"])[0])
    server = state["server"]
    if kind == "admit":
        gid = server.add_graph(state["graph"])[0]
        ticket = server.submit(gid, case["eps"], case["mu"])
        while server.pending:
            server.progress(wait=True)
        labels, stats = server.result(ticket, state["n"])
        server.remove_graph(gid)
        return {"labels": labels, "counts": {name: getattr(stats, name) for name in COUNTS[1:]}}
    tickets = [(server.submit(gid, eps, mu), n) for gid, n, eps, mu in state["queries"]]
    while server.pending:
        server.progress(wait=True)
    results = [server.result(ticket, n) for ticket, n in tickets]
    return {"labels": np.concatenate([r[0] for r in results]),
            "counts": np.array([[getattr(r[1], name) for name in COUNTS[1:]] for r in results], dtype=np.int64)}


def work(case):
    """The graph's rows and neighbour ids read once, the results written once;
    for a burst, once per query on the graphs' average size."""
    n = case["n"]
    if case["graph"] == "planted":
        m = n * (min(200.0, case["p_in"] * case["community"]) + 2 * case["inter"] + 0.1 * case["hubs"])
    else:
        m = 2 * case["edges"]
    if case["kind"] == "serve":
        share = sum(max(1000, n >> i) for i in range(case["graphs"])) / (case["graphs"] * n)
        return {"bytes": case["queries"] * share * (4.0 * m + 8 * n), "flops": 0}
    flags = m if case["kind"] in ("flags", "noalloc") else 0
    return {"bytes": 4.0 * m + 9 * n + flags, "flops": 0}
