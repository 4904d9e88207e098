"""Calls on contexts whose arena just holds what the launches' forms need, and
on arenas from there up: every call runs, whatever of the faster forms' scratch
(a team's blocks and list regions, the pairing's counts, row sizes by a bound,
the evaluators' partial sums) fits beside it, and gives the result of an ample
arena.  The smallest arena of each call is the peak of its launches' form."""
import math

import numpy as np
import pytest
import torch

import heipa
from graphs import block_weights, csr_from_arrays, random_partition
from test_gpu_parity import _dev

pytestmark = pytest.mark.gpu


def _leaves(n):
    return csr_from_arrays(n, np.arange(7, n), np.arange(7, n) ** 2 % 7)


GRAPHS = {
    "rgg50": lambda: heipa.gen_rgg(50, 4.0, 3, 9),
    "rgg1k": lambda: heipa.gen_rgg(1000, 8.0, 3, 9),
    "rgg16k": lambda: heipa.gen_rgg(16384, 8.0, 3, 9),
    "rgg140k": lambda: heipa.gen_rgg(140000, 6.0, 3, 9),
    "rmat12": lambda: heipa.gen_rmat(12, 0, 16.0, 0.57, 0.19, 0.19, 5, 10, False),
    "rmat16": lambda: heipa.gen_rmat(16, 0, 16.0, 0.57, 0.19, 0.19, 5, 10, False),
    "leaves300": lambda: _leaves(307),
    "leaves9k": lambda: _leaves(9007),
    "isolated70k": lambda: csr_from_arrays(70001, [0, 1], [1, 2]),
}
# (call, graph, blocks): arena bytes
CALLS = {
    ("cut", "rgg16k", 8): 256,
    ("cost", "rmat16", 8): 1024,
    ("weights", "rgg50", 8): 256,
    ("weights", "rmat16", 8): 256,
    ("match", "rgg50", 8): 1792,
    ("match", "leaves300", 8): 14592,
    ("match", "leaves9k", 8): 397824,
    ("match", "isolated70k", 8): 3641600,
    ("match", "rmat12", 8): 143616,
    ("refine", "rgg50", 2): 16384,
    ("refine", "rgg1k", 200): 418048,
    ("refine", "rgg16k", 64): 1524736,
    ("rebalance", "rgg16k", 64): 1524736,
    ("rebalance", "rmat12", 100): 561152,
    ("rebalance", "rgg140k", 64): 12863232,
    ("partition", "rgg1k", 2): 206592,
    ("partition", "rgg16k", 16): 2913024,
    ("im", "rgg1k", 8): 214784,
    ("hm", "rgg1k", 8): 222976,
}
EXTRA = [0, 1 << 12, 3 << 12, 1 << 15, 1 << 16, 3 << 16, 1 << 18, 1 << 20, 3 << 20]


def _call(c, call, g, dg, k):
    imbalance = 1.0005 if call == "rebalance" else 1.03
    part = random_partition(g.n, k, 7, 2.0 if call == "rebalance" else 0.0)
    pd = heipa.from_numpy_u32(part)
    if call == "cut":
        return c.edge_cut(dg, pd)
    if call == "cost":
        return c.comm_cost(dg, pd, torch.arange(k * k, dtype=torch.int32, device="cuda:0"), k)
    if call == "weights":
        bw, mx = c.block_weights(dg, pd, k)
        return bw.tolist(), mx
    if call == "match":
        mapping, nc, _ = c.match(dg)
        return heipa.to_numpy_u32(mapping).tobytes(), nc
    if call in ("refine", "rebalance"):
        lmax = math.ceil(imbalance * g.g_weight / k)
        cut, maxw, _ = c.jet_refine(dg, pd, k, lmax, False, 1, 10 ** 9, int(block_weights(g, part, k).max()))
        return heipa.to_numpy_u32(pd).tobytes(), cut, maxw
    if call == "partition":
        return heipa.to_numpy_u32(c.partition(dg, k, 0.03, 1, False)[0]).tobytes()
    if call == "im":
        return heipa.to_numpy_u32(c.im_partition(dg, [2, 4], [1, 10], 0.03, 1)[0]).tobytes()
    c.set_option(heipa.OPT_HM_WORKERS, 1)
    return heipa.to_numpy_u32(c.hm_partition(dg, [2, 4], 0.03, 1)).tobytes()


@pytest.mark.parametrize("call,graph,k", sorted(CALLS))
def test_scratch_limits(call, graph, k):
    g = GRAPHS[graph]()
    dg = _dev(g)
    need = CALLS[(call, graph, k)]
    got = []
    for arena in [1 << 30] + [need + x for x in EXTRA]:
        print(f"scratch {call} {graph} k={k} arena={arena}", flush=True)
        c = heipa.Context(0, arena)
        try:
            got.append(_call(c, call, g, dg, k))
        finally:
            c.close()
        assert got[-1] == got[0], arena
