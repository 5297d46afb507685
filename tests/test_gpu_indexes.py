"""The reverse-entry index of graphs large enough to be split into buckets
(over 2^21 entries): a pass writes the flags of both entries of every edge
through it, so they must equal the oracle's (needs an MI355X)."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_bind as ob
import efficientstructuralgraphclusteringongpus_amd as sgc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("extra", [0, 1, 40000])
def test_bucket_searches(ctx, extra):
    """2^20 + extra edges: communities, and hubs around the longest row a
    bucket takes (4096), linked with each other."""
    rng = np.random.default_rng(extra)
    n, edges = 160007, (1 << 20) + extra
    hubs = {0: 5000, 7: 4097, 150000: 4096, 150001: 4095, n - 1: 9000}
    ids = np.array(list(hubs))
    u = np.concatenate([np.full(d - len(hubs) + 1, h) for h, d in hubs.items()] + [np.repeat(ids, len(ids))])
    v = np.concatenate([rng.choice(np.setdiff1d(np.arange(n), ids), d - len(hubs) + 1, replace=False)
                        for d in hubs.values()] + [np.tile(ids, len(ids))])
    keys = np.unique((np.minimum(u, v) * n + np.maximum(u, v))[u != v])
    while len(keys) < edges:
        a = rng.integers(0, n, edges)
        b = np.where(rng.random(edges) < 0.8, a // 64 * 64 + rng.integers(0, 64, edges), rng.integers(0, n, edges))
        ok = (a != b) & (b < n) & ~np.isin(a, ids) & ~np.isin(b, ids)
        new = np.setdiff1d(np.minimum(a, b)[ok] * n + np.maximum(a, b)[ok], keys)
        keys = np.sort(np.concatenate([keys, rng.permutation(new)[:edges - len(keys)]]))
    g = sgc.HostGraph.from_edges(n, keys // n, keys % n)
    deg = np.diff(g.row_ptr)
    assert g.m == 2 * edges and [int(deg[h]) for h in hubs] == list(hubs.values())
    print("[case] m", g.m, "max degree", g.max_degree, flush=True)
    dg = sgc.DeviceGraph(ctx, g)
    try:
        for eps, mu in ((0.2, 3), (0.6, 2)):
            labels, core, sim, _ = ob.orc_scan(g.row_ptr, g.adj, eps, mu)
            r = sgc.scan(ctx, dg, eps, mu, want_sim=True)
            print("[case] eps", eps, "similar", r.stats.similar_edges, flush=True)
            assert np.array_equal(r.sim, sim) and np.array_equal(r.labels, labels) and np.array_equal(r.core, core)
    finally:
        dg.close()
