"""GPU parity of the team form of Jet (one launch of several workgroups on one
XCD runs whole iterations) at the sizes where its work split changes: levels
smaller than a wave, than the team, exactly one vertex per lane and just
beyond; degrees around the 32 that a rebuild keeps in registers; more than 64
blocks for the rows of wide vertices; hubs; resolve lists of up to 64 entries
(one wave) and longer.  Every traced iteration and the result must equal the
oracle's, bit for bit (integers: no tolerance)."""
import math

import numpy as np
import pytest

import heipa
import heipa_oracle as orc
from brute import vertex_weighted
from graphs import block_weights, csr_from_arrays, random_partition
from test_gpu_im import _D
from test_gpu_parity import GRAPHS, _dev, _trace_tuple

pytestmark = pytest.mark.gpu


def _regular(n, deg, wmod=9):
    """Every vertex has exactly `deg` neighbours (its nearest on a ring, and
    the opposite one if deg is odd; n even then)."""
    i = np.arange(n)
    us, vs = [], []
    for s in range(1, deg // 2 + 1):
        us.append(i)
        vs.append((i + s) % n)
    if deg % 2:
        us.append(i[:n // 2])
        vs.append(i[:n // 2] + n // 2)
    u, v = np.concatenate(us), np.concatenate(vs)
    return csr_from_arrays(n, u, v, 1 + (u * 7 + v * 13) % wmod)


CASES = {
    # name: (graph, k, skew of the starting partition, ultra)
    "one": (lambda: heipa.HostGraph(np.zeros(2, np.uint32), np.zeros(0, np.uint32)), 2, 0.0, False),
    "n17": (lambda: heipa.gen_rgg(17, 4.0, 3, 9), 3, 1.0, False),
    "n64": (lambda: heipa.gen_rgg(64, 6.0, 3, 9), 4, 2.0, True),
    "n4095": (lambda: heipa.gen_rgg(4095, 8.0, 3, 9), 64, 0.9, True),  # 16 vertices per wave
    "n16384": (lambda: heipa.gen_rgg(16384, 8.0, 3, 0), 23, 0.5, False),  # one vertex per lane of 256 waves
    "n16385": (lambda: heipa.gen_rgg(16385, 8.0, 3, 0), 7, 0.8, False),
    "n32769": (lambda: heipa.gen_rgg(32769, 8.0, 3, 100), 64, 0.3, False),  # a second sweep step
    "n50001": (lambda: heipa.gen_rgg(50001, 10.0, 3, 100), 100, 0.0, True),
    "deg31": (lambda: _regular(600, 31), 40, 0.7, True),
    "deg32": (lambda: _regular(600, 32), 40, 0.7, True),
    "deg33": (lambda: _regular(600, 33), 40, 0.7, True),
    "wide_k70": (lambda: heipa.gen_rmat(11, 0, 16.0, 0.57, 0.19, 0.19, 5, 10, False), 70, 0.8, True),
    "wide_k5": (lambda: _regular(900, 12), 5, 1.5, True),
    "hubs": (lambda: GRAPHS["hubs100"], 16, 0.6, False),
    "skewed": (lambda: heipa.gen_rmat(13, 0, 8.0, 0.57, 0.19, 0.19, 5, 10, False), 16, 1.0, False),
}


def _start(g, k, skew):
    part = (np.arange(g.n, dtype=np.int64) * k // max(g.n, 1)).astype(np.uint32)
    flip = np.random.default_rng(5).random(g.n) < 0.2
    return np.where(flip, random_partition(g.n, k, 11, skew), part).astype(np.uint32)


@pytest.fixture
def team(ctx):
    ctx.set_option(heipa.OPT_BLOCK_JET, 1 << 20)  # whole iterations per launch, however dense the level
    try:
        yield ctx
    finally:
        ctx.set_option(heipa.OPT_BLOCK_JET, 2048)


def _compare(gtr, otr, name):
    assert len(gtr) == len(otr), (name, len(gtr), len(otr))
    for i, (a, b) in enumerate(zip(gtr, otr)):
        assert _trace_tuple(a) == _trace_tuple(b), (name, i, _trace_tuple(a), _trace_tuple(b))


@pytest.mark.parametrize("name", sorted(CASES))
def test_team_jet(team, name):
    make, k, skew, ultra = CASES[name]
    g = make()
    part0 = _start(g, k, skew)
    lmax = math.ceil(1.03 * g.g_weight / k)
    cut0, maxw0 = orc.edge_cut(g, part0), int(block_weights(g, part0, k).max())
    print(f"team jet {name} n={g.n} m={g.m} k={k}", flush=True)
    op, ocut, omaxw, otr = orc.jet_refine(g, part0, k, lmax, ultra, 1, cut0, maxw0, trace_cap=4096)
    pd = heipa.from_numpy_u32(part0)
    gcut, gmaxw, gtr = team.jet_refine(_dev(g), pd, k, lmax, ultra, 1, cut0, maxw0, trace_cap=4096)
    _compare(gtr, otr, name)
    assert (gcut, gmaxw) == (ocut, omaxw)
    assert np.array_equal(heipa.to_numpy_u32(pd), op)


@pytest.mark.parametrize("hier", ["4:8:6", "2:3"])
@pytest.mark.parametrize("name", ["n64", "n16385", "deg31", "deg33", "wide_k5", "hubs"])
def test_team_map_refine(team, name, hier):
    """The mapping objective; with 2:3 most vertices have at least k neighbours
    and take the block-counter path."""
    g = CASES[name][0]()
    D, Dd = _D(*{"4:8:6": ([4, 8, 6], [1, 10, 100]), "2:3": ([2, 3], [7, 1])}[hier])
    k = D.shape[0]
    part0 = _start(g, k, 0.5)
    lmax = math.ceil(1.05 * g.g_weight / k)
    J0, maxw0 = orc.comm_cost(g, part0, D), int(block_weights(g, part0, k).max())
    print(f"team map {name} n={g.n} m={g.m} k={k}", flush=True)
    op, oJ, omaxw, otr = orc.map_refine(g, part0, D, lmax, J0, maxw0, trace_cap=4096)
    pd = heipa.from_numpy_u32(part0)
    gJ, gmaxw, gtr = team.map_refine(_dev(g), pd, Dd, k, lmax, 0, J0, maxw0, trace_cap=4096)
    _compare(gtr, otr, name)
    assert (gJ, gmaxw) == (oJ, omaxw)
    assert np.array_equal(heipa.to_numpy_u32(pd), op)


@pytest.fixture
def wide(ctx):
    """Every level runs as a team over all XCDs."""
    for opt, v in ((heipa.OPT_TEAM_JET, 0), (heipa.OPT_BLOCK_JET, 1), (heipa.OPT_WIDE_JET, 1 << 31)):
        ctx.set_option(opt, v)
    try:
        yield ctx
    finally:
        for opt, v in WIDE_DEFAULTS:
            ctx.set_option(opt, v)


WIDE_DEFAULTS = ((heipa.OPT_TEAM_JET, 1 << 15), (heipa.OPT_BLOCK_JET, 2048), (heipa.OPT_WIDE_JET, 0xFFFFFFFF))
WIDE_CASES = dict(CASES,
                  n131072=(lambda: heipa.gen_rgg(131072, 6.0, 3, 0), 12, 0.6, False),  # a vertex per lane of 2048 waves
                  n131073=(lambda: heipa.gen_rgg(131073, 6.0, 3, 9), 65, 0.6, False),
                  n262145=(lambda: heipa.gen_rgg(262145, 5.0, 3, 9), 33, 0.2, False),  # beyond one step of twice the waves
                  n270001=(lambda: heipa.gen_rgg(270001, 4.0, 3, 9), 5, 0.6, False))


@pytest.mark.parametrize("name", sorted(WIDE_CASES))
def test_wide_jet(wide, name):
    make, k, skew, ultra = WIDE_CASES[name]
    g = make()
    part0 = _start(g, k, skew)
    lmax = math.ceil(1.03 * g.g_weight / k)
    cut0, maxw0 = orc.edge_cut(g, part0), int(block_weights(g, part0, k).max())
    print(f"wide jet {name} n={g.n} m={g.m} k={k}", flush=True)
    op, ocut, omaxw, otr = orc.jet_refine(g, part0, k, lmax, ultra, 1, cut0, maxw0, trace_cap=4096)
    pd = heipa.from_numpy_u32(part0)
    gcut, gmaxw, gtr = wide.jet_refine(_dev(g), pd, k, lmax, ultra, 1, cut0, maxw0, trace_cap=4096)
    _compare(gtr, otr, name)
    assert (gcut, gmaxw) == (ocut, omaxw)
    assert np.array_equal(heipa.to_numpy_u32(pd), op)


@pytest.mark.parametrize("cap", [0, 16])
@pytest.mark.parametrize("name", ["n4095", "hubs", "skewed"])
def test_wide_stall(wide, name, cap):
    """Resolve lists beyond the LDS: the iteration ends on the device-wide path."""
    wide.set_option(heipa.OPT_RESOLVE_CAP, cap)
    try:
        test_wide_jet(wide, name)
    finally:
        wide.set_option(heipa.OPT_RESOLVE_CAP, 1 << 32)


@pytest.mark.parametrize("hier", ["4:8:6", "2:3"])
@pytest.mark.parametrize("name", ["n64", "n16385", "deg33", "wide_k5", "hubs"])
def test_wide_map_refine(wide, name, hier):
    test_team_map_refine(wide, name, hier)


def test_team_on_every_xcd():
    """Contexts use the device's XCDs in turn: nine of them, each its own team."""
    g = heipa.gen_rgg(3000, 8.0, 3, 9)
    want = orc.partition(g, 16, 0.03, 1, False)[0]
    dg = _dev(g)
    for _ in range(9):
        c = heipa.Context(0, 64 << 20)
        try:
            assert np.array_equal(heipa.to_numpy_u32(c.partition(dg, 16, 0.03, 1, False)[0]), want)
        finally:
            c.close()


def _twins(leaves, groups):
    """`leaves` vertices of degree 2 in `groups` interleaved groups of twins."""
    i = np.arange(leaves)
    a, b = i % groups, groups + (i % groups) * 7 % groups
    return csr_from_arrays(leaves + 2 * groups, np.concatenate([i + 2 * groups] * 2), np.concatenate([a, b]))


def _bipartite(leaves, hubs, deg, seed):
    """Vertices with `deg` random neighbours among `hubs` (of varied degree and edge weight)."""
    rng = np.random.default_rng(seed)
    v = np.concatenate([np.sort(rng.choice(hubs, deg, replace=False)) for _ in range(leaves)])
    u = hubs + np.repeat(np.arange(leaves), deg)
    return csr_from_arrays(hubs + leaves, u, v, 1 + (u + v) % 5)


MATCH = {
    "leaves": lambda: csr_from_arrays(9007, np.arange(7, 9007), np.arange(7, 9007) ** 2 % 7),  # all passes' first
    "relatives": lambda: _bipartite(6000, 300, 3, 1),  # few twins, the rest by their smallest neighbour
    "relatives_long": lambda: _bipartite(600, 140, 130, 2),  # keys by a wave each
    "twins": lambda: _twins(20000, 6),  # groups that span the members' shares
    "twins_many": lambda: _twins(5000, 1500),  # groups of 3 and 4
    "isolated": lambda: csr_from_arrays(40000, [0, 1], [1, 2]),  # one group of all but three
    "isolated_many": lambda: csr_from_arrays(70001, [0, 1], [1, 2]),  # longer than a team sorts
    "n1": lambda: heipa.HostGraph(np.zeros(2, np.uint32), np.zeros(0, np.uint32)),
    "n2": lambda: _regular(2, 1),
    "tile": lambda: _regular(16384, 4),  # one list entry per lane of 256 waves
    "tile_and_one": lambda: _regular(16385, 4),
    "list_limit": lambda: heipa.gen_rgg(65536, 6.0, 3, 0),  # the longest list a team takes over
    "beyond_list": lambda: heipa.gen_rgg(65537, 6.0, 3, 10),  # launches first, then a team
    "beyond_map": lambda: heipa.gen_rgg((1 << 18) + 1, 5.0, 3, 10),  # the mapping is the host's
    "wide": lambda: _regular(700, 130),  # adjacencies walked by a whole wave
    "dense": lambda: heipa.gen_rmat(15, 0, 24.0, 0.57, 0.19, 0.19, 5, 10, False),  # over 2^20 edges
    "hubs": lambda: GRAPHS["hubs100"],
}


@pytest.mark.parametrize("name", sorted(MATCH))
def test_team_match(ctx, name):
    """Matching where the rounds move from launches to a team, and within it."""
    g = MATCH[name]()
    print(f"team match {name} n={g.n} m={g.m}", flush=True)
    omp, onc, ost = orc.match(g, 12345)
    gmp, gnc, gst = ctx.match(_dev(g))
    assert gnc == onc
    assert np.array_equal(heipa.to_numpy_u32(gmp), omp)
    for f in ("rounds", "after_hem", "ran_leaf", "ran_twin", "ran_relative", "after_relative"):
        assert getattr(gst, f) == getattr(ost, f), f


def _overloaded(n, k, moved, eps, weighted):
    """Consecutive blocks, `moved` vertices of them in block 0 instead."""
    g = heipa.gen_rgg(n, 6.0, 3, 9)
    if weighted:
        g = vertex_weighted(g, 4, 40)
    part = (np.arange(n, dtype=np.int64) * k // n).astype(np.uint32)
    part[np.random.default_rng(1).choice(n, moved, replace=False)] = 0
    return g, part, math.ceil((1 + eps) * int(g.g_weight) / k)


@pytest.mark.parametrize("k,moved,eps,weighted", [(33, 300, 0.0005, True), (64, 40000, 0.0005, False),
                                                  (8, 300, 0.0005, False)])
def test_two_member_resolve(ctx, k, moved, eps, weighted):
    """Resolve lists of a level with two members per compute unit (more than
    512 vertices for each of 256): those that fit its 2048 entries are resolved
    in the launch, by weak and by strong rebalancing; only the longer ones go to
    the device-wide path, as often as in launches with the same capacity."""
    g, part0, lmax = _overloaded(140000, k, moved, eps, weighted)
    dg = _dev(g)
    cut0, maxw0 = ctx.edge_cut(dg, heipa.from_numpy_u32(part0)), int(block_weights(g, part0, k).max())
    print(f"two members k={k} moved={moved} eps={eps}", flush=True)

    def run(block_jet, cap):
        ctx.set_option(heipa.OPT_BLOCK_JET, block_jet)
        ctx.set_option(heipa.OPT_RESOLVE_CAP, cap)
        ctx.prof_enable(True)
        ctx.prof_filter("jet_rebalance_global")
        ctx.prof_reset()
        try:
            pd = heipa.from_numpy_u32(part0)
            cut, maxw, tr = ctx.jet_refine(dg, pd, k, lmax, False, 1, cut0, maxw0, trace_cap=4096)
            launches = ctx.prof_stats().get("jet_rebalance_global", {"launches": 0})["launches"]
        finally:
            ctx.prof_enable(False)
            ctx.prof_filter("")
            ctx.set_option(heipa.OPT_BLOCK_JET, 2048)
            ctx.set_option(heipa.OPT_RESOLVE_CAP, 1 << 32)
        return launches, (cut, maxw, heipa.to_numpy_u32(pd).tobytes(), [_trace_tuple(t) for t in tr])

    short, want = run(0, 64)
    long, same = run(0, 2048)
    assert same == want
    assert long < short and any(t[2] == 2 and t[4] > 64 for t in want[3])  # lists of 65 to 2048, strong ones too
    team, got = run(2048, 1 << 32)
    assert got == want
    assert team == long


ROWS = {
    # rows of wide vertices beyond 64 blocks: degrees around the 256 up to which
    # 16 lanes take one, lane groups on both sides of it, hubs, three and more words per mask
    "deg256": (lambda: _regular(1200, 256), 70),
    "deg257": (lambda: _regular(1200, 257), 70),
    "rmat_k65": (lambda: heipa.gen_rmat(12, 0, 40.0, 0.57, 0.19, 0.19, 5, 10, False), 65),
    "rmat_k97": (lambda: heipa.gen_rmat(13, 0, 30.0, 0.57, 0.19, 0.19, 5, 10, False), 97),
    "rmat_k200": (lambda: heipa.gen_rmat(14, 0, 30.0, 0.57, 0.19, 0.19, 5, 10, False), 200),
    "rgg_k66": (lambda: heipa.gen_rgg(20000, 90.0, 3, 10), 66),
}


def _rows(ctx, name, g, k, form):
    part0 = _start(g, k, 0.8)
    lmax = math.ceil(1.03 * g.g_weight / k)
    cut0, maxw0 = orc.edge_cut(g, part0), int(block_weights(g, part0, k).max())
    print(f"team rows {name} {form} n={g.n} m={g.m} k={k}", flush=True)
    op, ocut, omaxw, otr = orc.jet_refine(g, part0, k, lmax, False, 1, cut0, maxw0, trace_cap=4096)
    opts = {"one_xcd": ((heipa.OPT_BLOCK_JET, 1 << 20),), "all_xcds": ((heipa.OPT_TEAM_JET, 0), (heipa.OPT_BLOCK_JET, 1))}
    for opt, v in opts[form]:
        ctx.set_option(opt, v)
    try:
        pd = heipa.from_numpy_u32(part0)
        gcut, gmaxw, gtr = ctx.jet_refine(_dev(g), pd, k, lmax, False, 1, cut0, maxw0, trace_cap=4096)
    finally:
        for opt, v in WIDE_DEFAULTS:
            ctx.set_option(opt, v)
    _compare(gtr, otr, name)
    assert (gcut, gmaxw) == (ocut, omaxw)
    assert np.array_equal(heipa.to_numpy_u32(pd), op)


@pytest.mark.parametrize("form", ["one_xcd", "all_xcds"])
@pytest.mark.parametrize("name", sorted(ROWS))
def test_team_rows_many_blocks(ctx, name, form):
    make, k = ROWS[name]
    _rows(ctx, name, make(), k, form)


@pytest.mark.parametrize("form", ["one_xcd", "all_xcds"])
@pytest.mark.parametrize("deg", [4, 5, 32, 33])
@pytest.mark.parametrize("n", [40, 700, 20000])
def test_team_rows_few_blocks(ctx, n, deg, form):
    """Every vertex wide, few or many of them to a wave: rows by a lane or by 16."""
    _rows(ctx, f"n{n} deg{deg}", _regular(n, deg), 4, form)
