"""The framework's work that its performance is measured on.

Every case is one call of a public entry point of the Python binding (or one
batch through the pool) on synthetic graphs of the three families that the
tests and the benchmark use: 2D grids, random geometric graphs (RGG) and
R-MAT graphs.  Inputs are made from the seed alone.  The contexts and pools
are the handles that a program opens once and keeps.

    edge_cut    the smallest call: one evaluation of a given partition
    score       process-mapping cost J and block weights of a mapping
    match       one coarsening step's matching
    refine      Jet on a partition whose vertices have shifted a little, as a
                program calls it after its graph's load changed
    partition   a whole multilevel solve
    im, hm      the two process-mapping solvers
    pool        many graphs at once through the pool (batched form), or a
                queue of larger mixed requests (served form)
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gpu-heipa_amd", "python"))
import heipa  # noqa: E402

GIB = 1 << 30
DEVICE = "cuda:0"
_handles = {}


def _context():
    """The one context that a single-threaded program keeps."""
    if "ctx" not in _handles:
        _handles["ctx"] = heipa.Context(0, 8 * GIB)
    return _handles["ctx"]


def _pool(slots):
    if slots not in _handles:
        _handles[slots] = heipa.Pool(slots, 2 * GIB)
    return _handles[slots]


def listed():
    return [
        # a partition of a small graph is evaluated: latency of one call
        dict(name="cut-rgg14", kind="edge_cut", graph="rgg", n=16384, deg=8.0, wmod=10, k=16),
        # a 4:8:6 mapping of a skewed graph is scored: a bandwidth-sized call
        dict(name="score-rmat18", kind="score", graph="rmat", n=1 << 18, deg=16.0, wmod=100, hier="4:8:6"),
        # coarsening: one matching of the mesh-like and of the skewed family
        dict(name="match-rgg20", kind="match", graph="rgg", n=1 << 20, deg=12.0, wmod=10),
        dict(name="match-rmat-ragged", kind="match", graph="rmat", n=99991, deg=16.0, wmod=100),
        # refinement alone, on a graph of odd size with k that is no power of two
        dict(name="refine-rgg-k23", kind="refine", graph="rgg", n=130003, deg=12.0, wmod=100, k=23, ultra=True),
        # whole solves: the smallest, the mesh, the skewed one, the largest
        dict(name="part-rgg10-k8", kind="partition", graph="rgg", n=1500, deg=8.0, wmod=10, k=8, ultra=False),
        dict(name="part-grid512-k32", kind="partition", graph="grid", n=512 * 512, deg=4.0, wmod=0, k=32,
             ultra=False),
        dict(name="part-rmat-k16", kind="partition", graph="rmat", n=50000, deg=8.0, wmod=10, k=16, ultra=False),
        dict(name="part-rgg20-k64-ultra", kind="partition", graph="rgg", n=1 << 20, deg=12.0, wmod=10, k=64,
             ultra=True),
        # process mapping with the direct and with the recursive solver
        dict(name="im-rgg18-486", kind="im", graph="rgg", n=1 << 18, deg=12.0, wmod=10, hier="4:8:6"),
        dict(name="hm-rmat16-486", kind="hm", graph="rmat", n=1 << 16, deg=16.0, wmod=100, hier="4:8:6"),
        # the batched form's mix: small graphs of 10^3 to 6.5 * 10^4 vertices
        dict(name="pool-batched-32", kind="pool", mix="batched", count=32, slots=8),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["edge_cut", "score", "match", "refine", "partition", "partition", "partition", "im", "hm",
                       "pool"])
    if kind == "pool":
        if rng.random() < 0.7:
            return dict(kind=kind, mix="batched", count=rng.randint(8, 32), slots=8)
        return dict(kind=kind, mix="served", count=rng.randint(2, 5), slots=12)
    graph = rng.choice(["rgg", "rmat", "grid"] if kind != "hm" else ["rgg", "rmat"])
    skewed = graph == "rmat"
    top = {"edge_cut": 1 << 20, "score": 1 << 18, "match": 1 << 18 if skewed else 1 << 20,
           "refine": 1 << 15 if skewed else 1 << 18, "partition": 1 << 16 if skewed else 1 << 19,
           "im": 1 << 16 if skewed else 1 << 18, "hm": 1 << 16}[kind]
    n = _log_uniform(rng, {"im": 8000, "hm": 8000}.get(kind, 1024), top)
    c = dict(kind=kind, graph=graph, n=n, deg=4.0 if graph == "grid" else rng.choice([8.0, 12.0, 16.0]),
             wmod=0 if graph == "grid" else rng.choice([0, 10, 100]))
    if kind in ("score", "im", "hm"):
        c["hier"] = rng.choice(["4:8:6", "2:4:8"])
    if kind in ("edge_cut", "refine", "partition"):
        c["k"] = min(_log_uniform(rng, 2, 256), max(2, n // 64))
    if kind in ("refine", "partition"):
        # `ultra` runs 17 filter ratios instead of one
        c["ultra"] = not skewed and n <= 1 << 18 and c["k"] <= 64 and rng.random() < 0.4
    return c


def _host_graph(family, n, deg, wmod, seed):
    if family == "grid":
        side = max(2, int(round(math.sqrt(n))))
        return heipa.gen_grid(side, side)  # the solvers' own seed varies instead
    if family == "rgg":
        return heipa.gen_rgg(n, deg, 1000 + seed, wmod)
    return heipa.gen_rmat(max(1, math.ceil(math.log2(n))), n, deg, 0.57, 0.19, 0.19, 1000 + seed, wmod, False)


def _graph_of(case, seed):
    return _host_graph(case["graph"], case["n"], case["deg"], case["wmod"], seed)


def _hierarchy(case):
    hier = [int(x) for x in case["hier"].split(":")]
    return hier, [10 ** i for i in range(len(hier))]


def _random_part(n, k, seed):
    """Blocks of consecutive vertices, one vertex in eight elsewhere."""
    r = np.random.default_rng(seed)
    part = (np.arange(n, dtype=np.int64) * k // max(n, 1)).astype(np.uint32)
    move = r.random(n) < 0.125
    part[move] = r.integers(0, k, int(move.sum()), dtype=np.uint32)
    return part


def _requests(case, seed):
    """(graph, job arguments) of the batched or the served mix; the sizes are
    the case's, the graphs the seed's."""
    r = random.Random("%s %d" % (case["mix"], case["count"]))
    out = []
    for i in range(case["count"]):
        if case["mix"] == "batched":
            family, deg, wmod = r.choice([("rgg", 8.0, 10), ("rmat", 8.0, 10)])
            n, spec = _log_uniform(r, 1024, 65536), dict(k=r.choice([2, 4, 8, 16, 32]))
        else:
            family, deg, wmod = r.choice([("grid", 4.0, 0), ("rgg", 12.0, 100), ("rmat", 16.0, 100)])
            n = _log_uniform(r, 10000, 40000)
            spec = dict(k=r.randint(8, 256)) if r.random() < 0.7 else dict(hier=r.choice([[4, 8, 6], [2, 4, 8]]))
        out.append((_host_graph(family, n, deg, wmod, 100 * seed + i), spec))
    return out


def prepare(case, seed):
    kind = case["kind"]
    if kind == "pool":
        jobs = [(heipa.DeviceGraph(g, DEVICE), spec) for g, spec in _requests(case, seed)]
        parts = [torch.empty(g.n, dtype=torch.int32, device=DEVICE) for g, _ in jobs]
        return dict(kind=kind, pool=_pool(case["slots"]), jobs=jobs, parts=parts, seed=seed)
    host = _graph_of(case, seed)
    g = heipa.DeviceGraph(host, DEVICE)
    s = dict(kind=kind, ctx=_context(), g=g, seed=seed)
    if kind == "edge_cut":
        s["part"] = heipa.from_numpy_u32(_random_part(host.n, case["k"], seed))
    elif kind == "score":
        hier, dist = _hierarchy(case)
        D = heipa.distance_matrix(hier, dist)
        s.update(k=len(D), D=torch.from_numpy(D.reshape(-1)).to(DEVICE),
                 part=heipa.from_numpy_u32(_random_part(host.n, len(D), seed)))
    elif kind == "refine":
        # a balanced partition in which one vertex in fifty changed its block
        k = case["k"]
        part, st, _ = s["ctx"].partition(g, k, 0.03, 1, False)
        gen = torch.Generator(device="cpu").manual_seed(seed)
        move = (torch.rand(host.n, generator=gen) < 0.02).to(DEVICE)
        other = torch.randint(0, k, (host.n,), generator=gen, dtype=torch.int32).to(DEVICE)
        part = torch.where(move, other, part)
        s.update(k=k, ultra=case["ultra"], lmax=st.lmax, start=part, part=part.clone(),
                 cut=s["ctx"].edge_cut(g, part), maxw=s["ctx"].block_weights(g, part, k)[1],
                 bw=torch.empty(k, dtype=torch.int64, device=DEVICE))
    elif kind == "partition":
        s.update(k=case["k"], ultra=case["ultra"], part=torch.empty(host.n, dtype=torch.int32, device=DEVICE))
    elif kind in ("im", "hm"):
        hier, dist = _hierarchy(case)
        s.update(hier=hier, dist=dist, part=torch.empty(host.n, dtype=torch.int32, device=DEVICE))
    return s


def run(s):
    kind = s["kind"]
    if kind == "pool":
        jobs = [heipa.Pool.job(g, imbalance=0.03, seed=s["seed"], part=p, **spec)
                for (g, spec), p in zip(s["jobs"], s["parts"])]
        s["pool"].run(jobs)
        return dict(parts=s["parts"], cut=[j.cut for j in jobs][:16], status=sum(j.status for j in jobs))
    ctx, g = s["ctx"], s["g"]
    if kind == "edge_cut":
        return ctx.edge_cut(g, s["part"])
    if kind == "score":
        J = ctx.comm_cost(g, s["part"], s["D"], s["k"])
        bw, maxw = ctx.block_weights(g, s["part"], s["k"])
        return dict(J=J, bw=bw, maxw=maxw)
    if kind == "match":
        mapping, nc, _ = ctx.match(g, 12345 + s["seed"])
        return dict(mapping=mapping, nc=nc)
    if kind == "refine":
        s["part"].copy_(s["start"])
        cut, maxw, _ = ctx.jet_refine(g, s["part"], s["k"], s["lmax"], s["ultra"], 0, s["cut"], s["maxw"],
                                      bweights=s["bw"])
        return dict(part=s["part"], bw=s["bw"], cut=cut, maxw=maxw)
    if kind == "partition":
        part, st, _ = ctx.partition(g, s["k"], 0.03, s["seed"], s["ultra"], part=s["part"])
        return dict(part=part, cut=st.cut, maxw=st.maxw)
    if kind == "im":
        part, st, _ = ctx.im_partition(g, s["hier"], s["dist"], 0.03, s["seed"], part=s["part"])
        return dict(part=part, J=st.cut, maxw=st.maxw)
    return ctx.hm_partition(g, s["hier"], 0.03, s["seed"], False, part=s["part"])


def _graph_bytes(n, deg, wmod):
    """Offsets, both directions of every edge (RGG and grid: `deg` is the
    average degree; R-MAT: edges per vertex before duplicates go, about 0.9 of
    which stay) and their weights."""
    return 4 * (n + 1) + 4 * int(n * deg) * (2 if wmod else 1)


def work(case):
    if case["kind"] == "pool":
        mid, deg = (16000, 11.0) if case["mix"] == "batched" else (20000, 15.0)
        return dict(bytes=case["count"] * (_graph_bytes(mid, deg, 1) + 4 * mid), flops=0)
    n, deg = case["n"], case["deg"] * (1.8 if case["graph"] == "rmat" else 1.0)
    b = _graph_bytes(n, deg, case["wmod"]) + 4 * n  # the graph and one word per vertex (partition or map)
    if case["kind"] == "refine":
        b += 4 * n  # the partition comes and goes
    return dict(bytes=b, flops=0)


def exact(case, seed):
    """The evaluators' values; the solvers' results are partitions and maps,
    whole numbers that no closed form gives."""
    if case["kind"] not in ("edge_cut", "score"):
        return None
    g = _graph_of(case, seed)
    src = np.repeat(np.arange(g.n), np.diff(g.xadj.astype(np.int64)))
    w = np.ones(g.m, np.int64) if g.adjwgt is None else g.adjwgt.astype(np.int64)
    if case["kind"] == "edge_cut":
        part = _random_part(g.n, case["k"], seed)
        return int(w[part[src] != part[g.adjncy]].sum()) // 2
    hier, dist = _hierarchy(case)
    k = int(np.prod(hier))
    part = _random_part(g.n, k, seed)
    a, b = part[src].astype(np.int64), part[g.adjncy].astype(np.int64)
    d, size = np.zeros(g.m, np.int64), 1
    for h, x in zip(hier, dist):  # distance of the first level at which both lie in one group
        d = np.where(a // size != b // size, x, d)
        size *= h
    bw = np.bincount(part, minlength=k).astype(np.int64)
    return dict(J=int((w * d).sum()), bw=bw, maxw=int(bw.max()))
