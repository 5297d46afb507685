"""The exact counting kernels (every common neighbour counted at a serving
admission, early exits in out-of-core chips, which have no reverse-entry
index) against the oracle, at the sizes where the tables, rounds and segments
change (needs an MI355X).  All results are whole numbers: they must be equal."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_bind as ob
import efficientstructuralgraphclusteringongpus_amd as sgc

pytestmark = pytest.mark.gpu


def families(n, sizes, seed):
    """Families of six linked vertices around shared rows of the given sizes,
    their ids spread over all n."""
    rng = np.random.default_rng(seed)
    pool, src, dst, nxt = 7000, [], [], 7000
    for size in sizes:
        shared = rng.choice(pool, size=size, replace=False)
        members = np.arange(nxt, nxt + 6)
        nxt += 6
        for i, a in enumerate(members):
            kept = shared if i < 2 else shared[rng.random(size) >= rng.uniform(0, 0.6)]
            src.append(np.full(len(kept), a)), dst.append(kept)
            src.append(np.full(i, a)), dst.append(members[:i])
    ids = rng.choice(n - 2, size=nxt - 2, replace=False) + 1
    ids = np.concatenate([[0, n - 1], ids])  # the first and last bit of a bit set
    return sgc.HostGraph.from_edges(n, ids[np.concatenate(src)], ids[np.concatenate(dst)])


SIZES = (1, 9, 14, 15, 16, 17, 90, 91, 92, 95, 96, 97, 186, 187, 250, 251, 252, 1018, 1019, 1020, 1024,
         1530, 1531, 1532, 1536, 1537, 3066, 3067, 3072, 4607, 6900)


@pytest.mark.parametrize("n", [20001,             # small units: bit sets; two workgroups a CU for large ones
                               131072, 131073,    # ... and cuckoo hashes
                               458752, 458753,    # one workgroup a CU for large ones
                               1 << 20, (1 << 20) + 1])  # k_sim_units for large ones
def test_exact_kernels_match_oracle(ctx, n):
    g = families(n, SIZES, seed=n)
    print("[case] n", n, "m", g.m, "max degree", g.max_degree, flush=True)
    server = sgc.Server(ctx, sgc.Server.graph_bytes(g) + (1 << 20))
    try:
        gid = server.add_graph(g)[0]
        for eps, mu in ((0.2, 2), (0.5, 3), (0.8, 2)):
            labels, core, sim, _ = ob.orc_scan(g.row_ptr, g.adj, eps, mu)
            ticket = server.submit(gid, eps, mu)
            while server.pending:
                server.progress(wait=True)
            got, st = server.result(ticket, g.n)
            assert np.array_equal(got, labels) and st.similar_edges == int(sim.sum()) // 2, eps
            r, info = sgc.scan_ooc(ctx, g, eps, mu, sgc.ooc_min_budget(g, eps) + (1 << 20), want_sim=True)
            assert np.array_equal(r.sim, sim) and np.array_equal(r.labels, labels), eps
            print("[case] eps", eps, "similar", st.similar_edges, "chips", info.similarity_chips, flush=True)
    finally:
        server.close()


@pytest.mark.parametrize("batched", [False, True])
def test_queries_at_the_thresholds_of_edges(ctx, batched):
    """eps exactly at an edge's own (cn + 2) / sqrt((d(u) + 1) (d(v) + 1)),
    the doubles beside it, and just outside the band in which a query decides
    by the ratio alone; extreme eps."""
    g = sgc.HostGraph.rmat(11, 12, seed=4)
    rng = np.random.default_rng(5)
    rows = [set(g.adj[g.row_ptr[u]:g.row_ptr[u + 1]].tolist()) for u in range(g.n)]
    src = np.repeat(np.arange(g.n), np.diff(g.row_ptr).astype(np.int64))
    eps = [0.0, 1e-200, 1e200, 1.0]
    for k in rng.choice(g.m, 10, replace=False):
        u, v = int(src[k]), int(g.adj[k])
        e = (len(rows[u] & rows[v]) + 2) / np.sqrt(float(len(rows[u]) + 1) * float(len(rows[v]) + 1))
        eps += [float(e), float(np.nextafter(e, 0)), float(np.nextafter(e, 2)), float(e * (1 - 2e-6)), float(e * (1 + 2e-6))]
    server = sgc.Server(ctx, sgc.Server.graph_bytes(g) + (1 << 20))
    try:
        gid = server.add_graph(g)[0]
        server.set_batching(g.m if batched else 0)
        tickets = [server.submit(gid, e, 3) for e in eps]
        while server.pending:
            server.progress(wait=True)
        for e, t in zip(eps, tickets):
            labels, core, sim, _ = ob.orc_scan(g.row_ptr, g.adj, e, 3)
            got, st = server.result(t, g.n)
            assert np.array_equal(got, labels) and st.similar_edges == int(sim.sum()) // 2, e
        print("[case] batched", batched, "queries", len(eps), flush=True)
    finally:
        server.close()
