"""Compact row copies give way to the memory that passes and other graphs
need: with the device filled up to a chosen rest, what runs without the
copies still runs, with the same results (needs an MI355X)."""
from __future__ import annotations

import threading

import numpy as np
import pytest
import torch

import efficientstructuralgraphclusteringongpus_amd as sgc

pytestmark = pytest.mark.gpu


def say(*a):
    print("[case]", *a, flush=True)


def parts(g):
    """Bytes of a graph's CSR with each entry's row, of its indexes (two
    2^20-id windows), of a pass's work memory and of the compact row copies."""
    return 4 * g.n + 8 * g.m, 8 * g.m + 12 * g.n, 25 * g.m + 33 * g.n, 9 * g.m


def fill(ctx, rest):
    """Device memory taken until `rest` bytes are free."""
    torch.cuda.empty_cache()
    held = []
    for _ in range(8):
        free = ctx.memory()[0]
        say("free", free >> 20, "MB, down to", rest >> 20)
        if free <= rest + (32 << 20):
            break
        held.append(torch.empty(free - rest, dtype=torch.uint8, device="cuda"))
    return held


@pytest.fixture(scope="module")
def graph():
    g = sgc.HostGraph.rmat(21, 16, seed=7)
    say("n", g.n, "m", g.m)
    return g


@pytest.fixture(scope="module")
def expected(graph):
    with sgc.Context(0) as c:
        dg = sgc.DeviceGraph(c, graph)
        r = sgc.scan(c, dg, 0.4, 3)
        dg.close()
    return r.labels


def test_pass_comes_before_the_copies(graph, expected):
    held = None
    with sgc.Context(0) as c:
        csr, indexes, work, packed = parts(graph)
        try:
            held = fill(c, csr + indexes + work + packed // 2)
            dg = sgc.DeviceGraph(c, graph)
            try:
                assert np.array_equal(sgc.scan(c, dg, 0.4, 3).labels, expected)
            finally:
                dg.close()
        finally:
            del held
            torch.cuda.empty_cache()


def test_copies_are_given_back_for_another_graph(graph, expected):
    held = None
    with sgc.Context(0) as c:
        csr, _, _, packed = parts(graph)
        first = sgc.DeviceGraph(c, graph)
        second = None
        try:
            assert np.array_equal(sgc.scan(c, first, 0.4, 3).labels, expected)
            held = fill(c, csr - packed // 4)
            second = sgc.DeviceGraph(c, graph)
            for dg in (first, second):
                assert np.array_equal(sgc.scan(c, dg, 0.4, 3).labels, expected)
        finally:
            del held
            torch.cuda.empty_cache()
            if second:
                second.close()
            first.close()


def test_graphs_closed_in_any_order():
    g = sgc.HostGraph.rmat(10, 8, seed=3)
    with sgc.Context(0) as c:
        graphs = [sgc.DeviceGraph(c, g) for _ in range(3)]
        labels = sgc.scan(c, graphs[2], 0.5, 2).labels
        for i, left in ((1, (0, 2)), (2, (0,)), (0, ())):
            graphs[i].close()
            for k in left:
                assert np.array_equal(sgc.scan(c, graphs[k], 0.5, 2).labels, labels)


def test_graphs_freed_on_another_thread():
    """While the context's own thread uploads, scans and frees."""
    g = sgc.HostGraph.rmat(12, 8, seed=3)
    with sgc.Context(0) as c:
        own = sgc.DeviceGraph(c, g)
        labels = sgc.scan(c, own, 0.5, 2).labels
        for _ in range(4):
            others = [sgc.DeviceGraph(c, g) for _ in range(8)]
            freeing = threading.Thread(target=lambda: [dg.close() for dg in others])
            freeing.start()
            for _ in range(4):
                dg = sgc.DeviceGraph(c, g)
                assert np.array_equal(sgc.scan(c, dg, 0.5, 2).labels, labels)
                dg.close()
            freeing.join()
            assert np.array_equal(sgc.scan(c, own, 0.5, 2).labels, labels)
        own.close()
