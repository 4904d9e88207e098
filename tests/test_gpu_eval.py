"""The evaluators and the input checks share the edges out evenly over the
workgroups: rows that span several shares, shares whose source vertices do not
fit the offsets a workgroup holds at a time (2048), isolated vertices, and a
fault at any place of a share.  Values against numpy in 64 bits (integers: no
tolerance)."""
import ctypes

import numpy as np
import pytest
import torch

import heipa
from graphs import csr_from_arrays, random_partition
from test_gpu_parity import _dev

pytestmark = pytest.mark.gpu


def _sparse_ids():
    """200 edges among 60000 vertices: almost every vertex is isolated."""
    r = np.random.default_rng(3)
    return csr_from_arrays(60000, r.integers(0, 60000, 200), r.integers(0, 60000, 200), r.integers(1, 9, 200))


def _long_rows():
    """Three rows of 30000 entries: each spans many shares."""
    leaf = np.arange(3, 30003)
    return csr_from_arrays(30003, np.repeat([0, 1, 2], len(leaf)), np.tile(leaf, 3), 1 + np.arange(3 * len(leaf)) % 7)


CASES = {
    "sparse_ids": _sparse_ids,
    "long_rows": _long_rows,
    "one_edge": lambda: csr_from_arrays(2, [0], [1], [5]),
    "share": lambda: csr_from_arrays(512, np.arange(512), (np.arange(512) + 1) % 512),  # exactly 1024 edges
    "share_and_one": lambda: csr_from_arrays(600, np.arange(513), np.arange(513) + 1, 1 + np.arange(513)),
    "rmat": lambda: heipa.gen_rmat(14, 0, 16.0, 0.57, 0.19, 0.19, 3, 100, True),
}


def _sources(g):
    return np.repeat(np.arange(g.n), np.diff(g.xadj.astype(np.int64)))


@pytest.mark.parametrize("k", [3, 128, 129])  # D in LDS up to 128 blocks
@pytest.mark.parametrize("name", sorted(CASES))
def test_evaluators(ctx, name, k):
    g = CASES[name]()
    dg = _dev(g)
    part = random_partition(g.n, k, 7)
    pd = heipa.from_numpy_u32(part)
    src = _sources(g)
    w = np.ones(g.m, np.int64) if g.adjwgt is None else g.adjwgt.astype(np.int64)
    a, b = part[src].astype(np.int64), part[g.adjncy].astype(np.int64)
    D = np.random.default_rng(1).integers(0, 1000, (k, k)).astype(np.int32)
    print(f"eval {name} n={g.n} m={g.m} k={k}", flush=True)
    assert ctx.edge_cut(dg, pd) == int(w[a != b].sum()) // 2
    assert ctx.comm_cost(dg, pd, heipa.from_numpy_u32(D.reshape(-1).view(np.uint32)), k) == int((w * D[a, b]).sum())
    bw, mx = ctx.block_weights(dg, pd, k)
    vw = np.ones(g.n, np.int64) if g.vwgt is None else g.vwgt.astype(np.int64)
    want = np.bincount(part, weights=vw, minlength=k).astype(np.int64)
    assert np.array_equal(bw, want) and mx == want.max()


@pytest.mark.parametrize("fault", ["self_loop", "id", "weight"])
@pytest.mark.parametrize("where", [0, 1023, 1024, 29999, 30000, 45000, -1])
def test_faults_anywhere(ctx, fault, where):
    g = _long_rows()
    where %= g.m
    src = _sources(g)
    adj, ew = g.adjncy.copy(), g.adjwgt.copy()
    if fault == "self_loop":
        adj[where] = src[where]
    elif fault == "id":
        adj[where] = g.n
    else:
        ew[where] = 0
    bad = _dev(heipa.HostGraph(g.xadj, adj, ew, None))
    part = heipa.from_numpy_u32(random_partition(g.n, 4, 7))
    text = {"self_loop": "self loops", "id": "neighbour id", "weight": "edge weights"}[fault]
    for call in (lambda: ctx.edge_cut(bad, part), lambda: ctx.match(bad), lambda: ctx.block_weights(bad, part, 4)):
        with pytest.raises(heipa.HeipaError, match=text):
            call()


def test_block_id_out_of_range(ctx):
    g = _sparse_ids()
    dg = _dev(g)
    part = random_partition(g.n, 4, 7)
    part[g.n - 1] = 4
    pd = heipa.from_numpy_u32(part)
    D = heipa.from_numpy_u32(np.zeros(16, np.uint32))
    for call in (lambda: ctx.comm_cost(dg, pd, D, 4), lambda: ctx.block_weights(dg, pd, 4)):
        with pytest.raises(heipa.HeipaError, match="block id"):
            call()
    assert ctx.edge_cut(dg, pd) > 0  # an edge cut takes any block ids


@pytest.mark.parametrize("k", [4, 40000])  # staged in the context's pinned block, or beyond its size
def test_refused_block_weights_leave_the_output(ctx, k):
    g = _sparse_ids()
    dg = _dev(g)
    part = random_partition(g.n, k, 7)
    part[17] = k
    pd = heipa.from_numpy_u32(part)
    bw, maxw = np.full(k, -7, np.int64), ctypes.c_int64(-9)
    rc = ctx.L.heipa_block_weights(ctx.h, ctypes.byref(dg.desc), pd.data_ptr(), k,
                                   bw.ctypes.data_as(ctypes.POINTER(ctypes.c_int64)), ctypes.byref(maxw))
    assert rc == heipa.ERR_INVALID
    assert (bw == -7).all() and maxw.value == -9


def test_missing_arrays_are_refused(ctx):
    """A null partition, and a graph that claims edges without having vertices
    or arrays: refused before anything reaches the device."""
    g = _dev(_sparse_ids())
    bw, out = (ctypes.c_int64 * 4)(), ctypes.c_int64()
    assert ctx.L.heipa_block_weights(ctx.h, ctypes.byref(g.desc), None, 4, bw, None) == heipa.ERR_INVALID
    empty = heipa.Graph(0, 5, 0, heipa.UNIFORM_EW | heipa.UNIFORM_VW, 0, None, None, None, None)
    assert ctx.L.heipa_edge_cut(ctx.h, ctypes.byref(empty), None, ctypes.byref(out)) == heipa.ERR_INVALID
    assert ctx.L.heipa_block_weights(ctx.h, ctypes.byref(empty), None, 4, bw, None) == heipa.ERR_INVALID
    none = heipa.Graph(0, 0, 0, heipa.UNIFORM_EW | heipa.UNIFORM_VW, 0, None, None, None, None)
    assert ctx.L.heipa_edge_cut(ctx.h, ctypes.byref(none), None, ctypes.byref(out)) == heipa.OK and out.value == 0
    assert ctx.L.heipa_block_weights(ctx.h, ctypes.byref(none), None, 4, bw, None) == heipa.OK and list(bw) == [0] * 4


def test_edge_offsets_near_the_limit(ctx):
    """4294966296 directed edges, the last offsets within one stride of 2^32:
    every vertex but vertex 0 has all its edges to vertex 0 (made on the device)."""
    n, m = 1025, 2 ** 32 - 1000
    xadj = np.concatenate([[0], np.arange(n, dtype=np.uint64) * m // (n - 1)]).astype(np.uint32)
    adj = torch.zeros(m, dtype=torch.int32, device="cuda:0")
    xd = heipa.from_numpy_u32(xadj)
    g = heipa.Graph(n, m, n, heipa.UNIFORM_EW | heipa.UNIFORM_VW, 0, xd.data_ptr(), adj.data_ptr(), None, None)
    part = np.arange(n, dtype=np.uint32) % 3
    pd = heipa.from_numpy_u32(part)
    D = np.random.default_rng(1).integers(0, 1000, (3, 3)).astype(np.int32)
    Dd = heipa.from_numpy_u32(D.reshape(-1).view(np.uint32))
    deg = np.diff(xadj.astype(np.int64))
    print(f"eval m={m}", flush=True)
    torch.cuda.synchronize()
    out = ctypes.c_int64()
    assert ctx.L.heipa_edge_cut(ctx.h, ctypes.byref(g), pd.data_ptr(), ctypes.byref(out)) == heipa.OK
    assert out.value == int(deg[part != part[0]].sum()) // 2
    assert ctx.L.heipa_comm_cost(ctx.h, ctypes.byref(g), pd.data_ptr(), Dd.data_ptr(), 3, ctypes.byref(out)) == heipa.OK
    assert out.value == int((deg * D[part, part[0]].astype(np.int64)).sum())
