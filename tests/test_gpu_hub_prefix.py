"""Counts that use the first rows of a larger set of hub bitmaps (GPU): the
graph's rows are built for every vertex, then thresholds rise past all degrees
and fall again, in degree order and through the map of the original ids."""
import pytest

from patterns import C5, HOUSE

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode", ["unique", "reference"])
@pytest.mark.parametrize("pattern", [HOUSE, C5])
def test_thresholds_after_a_full_set(gat, gpu, mode, pattern):
    g = gat.Graph.rmat(10, 12, 0.57, 0.19, 0.19, 4)
    plan = gat.Plan(g, [pattern], mode)
    want, _ = plan.count({"hub_degree": -1})
    top = g.max_degree()
    for thr in (1, 9, 0, 64, 256, top, top + 1, 100000, 3, 0):
        for extra in ({}, {"slot_capacity": 16, "split_us": 1}):
            assert plan.count(dict(extra, hub_degree=thr))[0] == want, (thr, extra)
