"""The filter stage of the similarity phase (packed rows, LDS bit filters)
against the exact kernels alone and against the oracle, at the sizes where
its row layouts, owner tiers and units change (needs an MI355X).  All results
are whole numbers: they must be equal."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_bind as ob
import efficientstructuralgraphclusteringongpus_amd as sgc

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


def edge_graph(sizes, fans, seed):
    """Families of six linked vertices that share `size` pool vertices, each
    dropping up to 60 % of them (similar and dissimilar edges on both sides of
    the threshold), and fans: a centre with `d` low-degree leaves, which owns
    all its edges."""
    rng = np.random.default_rng(seed)
    pool, src, dst, nxt = 5000, [], [], 5000
    for size in sizes:
        shared = rng.choice(pool, size=size, replace=False)
        members = np.arange(nxt, nxt + 6)
        nxt += 6
        for i, a in enumerate(members):
            kept = shared if i < 2 else shared[rng.random(size) >= rng.uniform(0, 0.6)]
            src.append(np.full(len(kept), a)), dst.append(kept)
            src.append(np.full(i, a)), dst.append(members[:i])
    for d in fans:
        leaves = np.arange(nxt + 1, nxt + 1 + d)
        src.append(np.full(d, nxt)), dst.append(leaves)
        for _ in range(14):
            src.append(leaves), dst.append(rng.permutation(leaves))
        nxt += 1 + d
    return sgc.HostGraph.from_edges(nxt, np.concatenate(src), np.concatenate(dst))


@pytest.mark.parametrize("sizes,fans", [
    ((1, 2, 5, 6, 7, 8, 13, 14, 15, 58, 62, 63, 64, 65), (63, 64, 65, 128)),  # groups of 7, batches of 64 edges
    ((500, 505, 506, 507, 508, 511, 512, 513), (255, 256, 257, 511, 512, 513)),  # wave tier, wide rows
    ((1018, 1019, 1024, 2042, 2043, 2044, 2049), (700, 1030)),  # exact small tier, workgroup filter
    ((4000, 4990), (2047, 2048, 2049, 3000)),  # large filter
])
def test_filter_matches_exact_kernels_and_oracle(ctx, sizes, fans):
    g = edge_graph(sizes, fans, seed=sizes[-1])
    say("sizes", sizes, "fans", fans, "n", g.n, "m", g.m, "max degree", g.max_degree)
    dg = sgc.DeviceGraph(ctx, g)
    try:
        for eps, mu in ((0.1, 3), (0.2, 2), (0.5, 3), (0.75, 2), (0.95, 2)):
            dg.tuning = sgc.Tuning()
            r = sgc.scan(ctx, dg, eps, mu, want_sim=True)
            dg.tuning = sgc.Tuning(hash_tables=0)  # no filter stage
            x = sgc.scan(ctx, dg, eps, mu, want_sim=True)
            labels, core, sim, _ = ob.orc_scan(g.row_ptr, g.adj, eps, mu)
            assert np.array_equal(r.sim, sim) and np.array_equal(x.sim, sim), eps
            assert np.array_equal(r.core, core) and np.array_equal(r.labels, labels), eps
            assert r.stats.u_edges == x.stats.u_edges
            say("eps", eps, "similar", int(sim.sum()) // 2, "undecided", r.stats.u_edges)
    finally:
        dg.close()


@pytest.mark.parametrize("eps", [0.01, 0.02])
def test_similar_edges_of_long_rows_are_not_read_in_full(ctx, eps):
    """At low eps an edge between two rows of 4000 entries is similar after
    about 90 common neighbours: no filter reads the row first.  Short rows are
    read once at most."""
    g = edge_graph((4000, 4990), (), seed=8)
    deg = np.diff(g.row_ptr).astype(np.int64)
    src = np.repeat(np.arange(g.n), deg)
    lo, hi = np.minimum(deg[src], deg[g.adj]), np.maximum(deg[src], deg[g.adj])
    left = (src < g.adj) & (lo + 1 >= (hi + 1) * eps * eps) & (eps * eps * (lo + 1) * (hi + 1) > 4)
    long, short = int(lo[left & (lo > 1024)].sum()), int(lo[left & (lo <= 1024)].sum())
    dg = sgc.DeviceGraph(ctx, g)
    try:
        r = sgc.scan(ctx, dg, eps, 3, want_sim=True)
        labels, _, sim, _ = ob.orc_scan(g.row_ptr, g.adj, eps, 3)
        say("eps", eps, "long rows", long, "short rows", short, "loaded", r.stats.loaded_elements)
        assert np.array_equal(r.sim, sim) and np.array_equal(r.labels, labels)
        assert r.stats.loaded_elements < short + long / 2
    finally:
        dg.close()


@pytest.mark.parametrize("n,deg", [(40, 39), (3000, 900)])
def test_filter_on_one_degree_class(ctx, n, deg):
    """Regular rows: every vertex has (nearly) the same degree, so the classes
    are cut by the hash alone."""
    rng = np.random.default_rng(n)
    i = np.arange(n)
    offs = rng.choice(np.arange(1, (n + 1) // 2), size=min(deg // 2, (n - 1) // 2), replace=False)
    g = sgc.HostGraph.from_edges(n, np.concatenate([i for _ in offs]), np.concatenate([(i + o) % n for o in offs]))
    say("regular", g.n, g.m, g.max_degree)
    dg = sgc.DeviceGraph(ctx, g)
    try:
        for eps in (0.2, 0.3, 0.6):
            r = sgc.scan(ctx, dg, eps, 3, want_sim=True)
            _, _, sim, _ = ob.orc_scan(g.row_ptr, g.adj, eps, 3)
            assert np.array_equal(r.sim, sim)
    finally:
        dg.close()
