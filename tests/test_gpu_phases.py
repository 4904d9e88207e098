"""The phase times of a solve: the projections' time is in ms_uncontraction.
The two finest projections of 2^26 vertices without edges (every level halves)
read a map and a partition and write one: 10 bytes a vertex, which at 8 TB/s, the
nominal rate of the memory, take 126 us; queueing all projections takes less."""
import numpy as np
import pytest

import heipa

pytestmark = pytest.mark.gpu


def test_projection_time():
    n = 1 << 26
    dg = heipa.DeviceGraph(heipa.HostGraph(np.zeros(n + 1, np.uint32), np.zeros(0, np.uint32)))
    c = heipa.Context(0, 32 << 30)
    try:
        print(f"phases n={n}", flush=True)
        c.partition(dg, 2, 0.03, 1, False)
        st = min((c.partition(dg, 2, 0.03, 1, False)[1] for _ in range(3)), key=lambda st: st.ms_uncontraction)
    finally:
        c.close()
    print(f"uncontraction {st.ms_uncontraction:.3f} ms of {st.levels} levels", flush=True)
    assert st.ms_uncontraction >= 10.0 * n * 1.5 / 8e12 * 1e3
    assert st.ms_refinement > 0.0
