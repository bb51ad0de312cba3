"""Plans of which some leaf counts are kept in tables and others swept (GPU), on
graphs between the bounds of the choice, against the walk without tables (the
one of accounted counts)."""
import pytest

from patterns import C5, HOUSE, connected_patterns

pytestmark = pytest.mark.gpu


# mean neighbour degree 25 (edges of whole lists), 41 (truncated ones too), 61 (pools
# of one vertex) and, of R-MAT, above 64 (sums; pools keyed by the edge)
@pytest.mark.parametrize("graph", ["er20k", "er20k dense", "er3k", "rmat11"])
@pytest.mark.parametrize("mode", ["unique", "reference"])
def test_counts(gat, gpu, graph, mode):
    from graphautotune_amd._lib import GatError
    g = {"er20k": lambda: gat.Graph.erdos_renyi(20000, 24 / 20000, 3),
         "er20k dense": lambda: gat.Graph.erdos_renyi(20000, 40 / 20000, 3),
         "er3k": lambda: gat.Graph.erdos_renyi(3000, 60 / 3000, 3),
         "rmat11": lambda: gat.Graph.rmat(11, 8, 0.57, 0.19, 0.19, 6)}[graph]()
    five = connected_patterns(5)
    pats, want = [], []
    for p in [C5, HOUSE] + [five[i] for i in (0, 3, 6, 8, 10, 12, 14)]:
        try:
            plan = gat.Plan(g, [p], mode)
        except GatError:
            continue  # the reference has no defined value
        w, _ = plan.count(account=True)
        pats.append(p)
        want += w
        for cfg in ({}, {"split_us": 1, "queue_chunk": 1}, {"slot_capacity": 16}):
            assert plan.count(cfg)[0] == w, (p, cfg)
    assert len(pats) >= 6
    if mode == "unique":
        batched = gat.Plan(g, pats, mode)
        for cfg in ({}, {"split_us": 1, "slot_capacity": 16}):
            assert batched.count(cfg)[0] == want, cfg
