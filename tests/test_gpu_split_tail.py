"""A count of one root edge is a tail from its start: its wave hands on a long
rest as soon as the pace shows it, without waiting for the split budget (GPU).
The budget is half of what the edge takes unsplit, so a main launch that waits
for it takes at least that long."""
import numpy as np
import pytest

from patterns import C5

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["unique", "reference"])  # the pair sweep, and the walk above a leaf
def test_long_rest_is_handed_on_before_the_budget(gat, gpu, mode):
    g = gat.Graph.chung_lu(100003, 24.0, 2.1, 5000, 1)
    off, adj = (np.asarray(a) for a in g.csr())
    plan = gat.Plan(g, [C5], mode)
    if mode == "unique":  # degree order: the first entry of a light vertex's row is its heaviest neighbour
        e = int(plan.run_offsets()[50000])
    else:  # v1 < v0: from a light vertex to its heaviest smaller neighbour
        deg = np.diff(off)
        src = np.repeat(np.arange(len(deg)), deg)
        ok = (adj < src) & (deg[src] <= 16)
        e = int(np.flatnonzero(ok)[np.argmax(deg[adj[ok]])])
    plan.count_shard_edges(e, e + 1)  # tables and bitmaps are built here
    want, alone = plan.count_shard_edges(e, e + 1, {"split_us": -1})
    budget_ms = alone["main_kernel_ms"] / 2
    assert alone["split_tasks"] == 0 and budget_ms > 0.5, alone
    got, st = plan.count_shard_edges(e, e + 1, {"split_us": int(budget_ms * 1e3)})
    assert got == want
    assert st["main_kernel_ms"] < budget_ms and st["split_tasks"] > 0, (budget_ms, st)
