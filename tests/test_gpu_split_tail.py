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


def test_sum_over_the_father_is_split(gat, gpu):
    """A leaf whose count is summed over the father set of one edge between two
    hubs (about 7 of the 29 ms that one wave takes): its entries go to several
    waves, in the LDS launches and, with small set buffers, in the HBM launch."""
    pattern = "0010100011100110110111110"
    g = gat.Graph.chung_lu(300007, 24.0, 2.1, 20000, 1)
    plan = gat.Plan(g, [pattern], "unique")
    e = int(plan.run_offsets()[1000])
    plan.count_shard_edges(e, e + 1)
    want, alone = plan.count_shard_edges(e, e + 1, {"split_us": -1})
    budget_ms = alone["main_kernel_ms"] / 8
    assert alone["overflow_tasks"] == 0
    got, st = plan.count_shard_edges(e, e + 1, {"split_us": int(budget_ms * 1e3)})
    assert got == want
    assert st["main_kernel_ms"] < budget_ms, (budget_ms, st)
    for us in (1, 100, 2000):
        got, st = plan.count_shard_edges(e, e + 1, {"split_us": us, "slot_capacity": 16})
        assert got == want and st["overflow_tasks"] == 1 and st["split_tasks"] > 0, (us, got, st)
