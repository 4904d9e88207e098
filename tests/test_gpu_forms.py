"""The rebalancing corner cases of the launches' tests in the form that runs
every level as a team over all XCDs, and up to the most blocks that a team takes
(1200: the eviction bounds of more than 1024 are in device memory).  Every traced
iteration and the result must equal the oracle's, bit for bit."""
import math

import numpy as np
import pytest

import heipa
import heipa_oracle as orc
from graphs import block_weights, random_partition
from test_gpu_jet_edges import CASES, LARGE_K, MAP_HIERS, _same
from test_gpu_parity import _dev

pytestmark = pytest.mark.gpu


@pytest.fixture
def wide(ctx):
    ctx.set_option(heipa.OPT_TEAM_JET, 0)
    ctx.set_option(heipa.OPT_BLOCK_JET, 1)
    try:
        yield ctx
    finally:
        ctx.set_option(heipa.OPT_TEAM_JET, 1 << 15)
        ctx.set_option(heipa.OPT_BLOCK_JET, 2048)


def _refine(c, name, g, part0, k, lmax, ultra, level):
    cut0, maxw0 = orc.edge_cut(g, part0), int(block_weights(g, part0, k).max())
    print(f"wide form {name} ultra={ultra} level={level} n={g.n} k={k}", flush=True)
    op, ocut, omaxw, otr = orc.jet_refine(g, part0, k, lmax, ultra, level, cut0, maxw0, trace_cap=8192)
    pd = heipa.from_numpy_u32(part0)
    gcut, gmaxw, gtr = c.jet_refine(_dev(g), pd, k, lmax, ultra, level, cut0, maxw0, trace_cap=8192)
    _same(name, gtr, otr)
    assert (gcut, gmaxw) == (ocut, omaxw)
    assert np.array_equal(heipa.to_numpy_u32(pd), op), name


@pytest.mark.parametrize("ultra,level", [(False, 0), (False, 1), (True, 0)])
@pytest.mark.parametrize("name", sorted(CASES))
def test_wide_edges(wide, name, ultra, level):
    g, part0, k, lmax = CASES[name]
    _refine(wide, name, g, part0, k, lmax, ultra, level)


@pytest.mark.parametrize("name", sorted(CASES))
def test_wide_map_edges(wide, name):
    g, part0, k, lmax = CASES[name]
    D = orc.distance_matrix(*MAP_HIERS[k])
    Dd = heipa.from_numpy_u32(D.reshape(-1).view(np.uint32))
    J0, maxw0 = orc.comm_cost(g, part0, D), int(block_weights(g, part0, k).max())
    print(f"wide form map {name}", flush=True)
    op, oJ, omaxw, otr = orc.map_refine(g, part0, D, lmax, J0, maxw0, trace_cap=4096)
    pd = heipa.from_numpy_u32(part0)
    gJ, gmaxw, gtr = wide.map_refine(_dev(g), pd, Dd, k, lmax, 0, J0, maxw0, trace_cap=4096)
    _same(name, gtr, otr)
    assert (gJ, gmaxw) == (oJ, omaxw)
    assert np.array_equal(heipa.to_numpy_u32(pd), op), name


@pytest.mark.parametrize("k", [700, 1030, 1200])
def test_wide_large_k(wide, k):
    g = LARGE_K
    part0 = (np.arange(g.n, dtype=np.int64) * k // g.n).astype(np.uint32)
    flip = np.random.default_rng(5).random(g.n) < 0.15
    part0 = np.where(flip, random_partition(g.n, k, 11, 0.3), part0).astype(np.uint32)
    _refine(wide, f"k{k}", g, part0, k, math.ceil(1.03 * g.n / k), False, 0)
