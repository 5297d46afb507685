"""What a serving engine charges a graph's query slots against its memory
budget covers what the slots hold (host arithmetic only, no GPU)."""
from __future__ import annotations

import os
import re

import pytest

import efficientstructuralgraphclusteringongpus_amd as sgc

HEADER = os.path.join(os.path.dirname(sgc.__file__), "csrc", "device.h")


def counter_bytes():
    """Size of a pass's counter buffer, from its layout in the header."""
    text = open(HEADER).read()
    first, stripes, slots = (int(re.search(rf"\b{name} = (\d+)", text).group(1))
                             for name in ("kStripe0", "kStripes", "kStripeSlots"))
    assert re.search(r"kCntWords = kStripe0 \+ kStripes \* kStripeSlots", text)
    return 8 * (first + stripes * slots)


@pytest.mark.parametrize("n", [2, 1000, 5000])
def test_a_slot_is_charged_for_its_arrays_and_counters(n):
    g = sgc.HostGraph.from_edges(n, list(range(n - 1)), list(range(1, n)))
    slot = sgc.Server.graph_bytes(g, 5) - sgc.Server.graph_bytes(g, 4)
    # flags, five words and a byte a vertex, the counters
    assert slot >= g.m + 21 * g.n + counter_bytes()
