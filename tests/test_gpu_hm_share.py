"""Multisection whose workers share the subtrees' children: more workers than
subtrees of the first split, fewer, and worker arenas that hold some of the
subtrees and not others (those are handed back whole).  The mapping must be
the oracle's, bit for bit (integers: no tolerance)."""
import numpy as np
import pytest

import heipa
import heipa_oracle as orc
from test_gpu_parity import _dev

pytestmark = pytest.mark.gpu

HIERS = {"3:4:2": [3, 4, 2], "2:3:2:3": [2, 3, 2, 3], "5:4": [5, 4]}


@pytest.fixture(scope="module")
def case():
    g = heipa.gen_rmat(12, 0, 12.0, 0.57, 0.19, 0.19, 11, 50, False)  # the first split's subtrees differ widely
    return g, {name: orc.hm_partition(g, h, 0.03, 1, False) for name, h in HIERS.items()}


@pytest.mark.parametrize("worker_bytes", [0, 3 << 20])
@pytest.mark.parametrize("workers", [2, 3, 8])
@pytest.mark.parametrize("hier", sorted(HIERS))
def test_hm_shared_subtrees(ctx, case, hier, workers, worker_bytes):
    g, want = case
    dg = _dev(g)
    print(f"hm {hier} workers={workers} bytes={worker_bytes}", flush=True)
    ctx.set_option(heipa.OPT_HM_WORKERS, workers)
    ctx.set_option(heipa.OPT_HM_WORKER_BYTES, worker_bytes)
    try:
        for _ in range(2):
            part = ctx.hm_partition(dg, HIERS[hier], 0.03, 1, False)
            assert np.array_equal(heipa.to_numpy_u32(part), want[hier])
    finally:
        ctx.set_option(heipa.OPT_HM_WORKERS, 8)
        ctx.set_option(heipa.OPT_HM_WORKER_BYTES, 0)


@pytest.mark.parametrize("share,workers", [(0.4, 2), (0.15, 3), (0.02, 6)])
def test_hm_worker_memory(ctx, case, share, workers):
    """Arenas of the given share of the free device memory, three subtrees of
    the first split and six of the second: workers that cannot be opened
    leave the others, those beyond the three stay within an eighth of the free
    memory, and a later call uses the ones that the first call opened."""
    import torch
    g, want = case
    dg = _dev(g)
    ctx.set_option(heipa.OPT_HM_WORKERS, 0)  # none kept from earlier calls
    ctx.set_option(heipa.OPT_HM_WORKERS, 8)
    free = torch.cuda.mem_get_info()[0]
    ctx.set_option(heipa.OPT_HM_WORKER_BYTES, int(share * free))
    print(f"hm worker memory {share}", flush=True)
    try:
        for _ in range(2):
            part = ctx.hm_partition(dg, HIERS["2:3:2:3"], 0.03, 1, False)
            assert np.array_equal(heipa.to_numpy_u32(part), want["2:3:2:3"])
            held = (free - torch.cuda.mem_get_info()[0]) / free
            assert abs(held - share * workers) < 0.01
    finally:
        ctx.set_option(heipa.OPT_HM_WORKER_BYTES, 0)
        ctx.set_option(heipa.OPT_HM_WORKERS, 8)
