"""COUNT values kept in tables within a count (array store, GPU): the edge
tables, the pools keyed by the first vertex, the second or the root edge, and
the sweep of the last two levels together. Counts against the oracle where the
tables end inside the graph, where keys share a table, and under splitting,
overflow, replays and many counts in a row (each has its own epoch)."""
import pytest

from patterns import C5, HOUSE, connected_patterns

pytestmark = pytest.mark.gpu

K23 = "0011100111110001100011000"  # complete bipartite 2 x 3


def edges_pattern(n, edges):
    return "".join("1" if (i, j) in edges or (j, i) in edges else "0" for i in range(n) for j in range(n))


def cycle(n):
    return edges_pattern(n, {(i, (i + 1) % n) for i in range(n)})


def path(n):
    return edges_pattern(n, {(i, i + 1) for i in range(n - 1)})


CONFIGS = ({}, {"split_us": 1, "queue_chunk": 1}, {"slot_capacity": 16, "hub_degree": 8, "split_us": -1},
           {"hub_degree": -1, "search_linear_threshold": 8, "queue_chunk": 3})


@pytest.fixture(scope="module")
def graphs(gat):
    return {"rmat8": gat.Graph.rmat(8, 6, 0.57, 0.19, 0.19, 3), "cl300": gat.Graph.chung_lu(300, 8.0, 2.1, 60, 5),
            "er60": gat.Graph.erdos_renyi(60, 0.15, 2)}


@pytest.mark.parametrize("gname", ["rmat8", "cl300", "er60"])
@pytest.mark.parametrize("mode", ["unique", "reference"])
def test_patterns_and_configs(gat, orc, gpu, graphs, gname, mode):
    from graphautotune_amd._lib import ScheduleData, GatError
    g = graphs[gname]
    off, adj = g.csr()
    pats = [C5, HOUSE, K23, path(5)] + list(connected_patterns(5))[::4]
    if gname == "er60":
        pats += [cycle(6), path(6)] + list(connected_patterns(6))[:: 12 if mode == "unique" else 40]
    for p in pats:
        try:
            plan = gat.Plan(g, [p], mode)
        except GatError:
            continue  # reference mode: the reference has no defined value
        if mode == "unique":
            want = orc.unique_count(off, adj, p)
        else:
            want, ok = orc.reference_count(off, adj, orc.schedule(p, ScheduleData))
            assert ok
        for cfg in CONFIGS:
            got, _ = plan.count(cfg)
            assert got == [want], (gname, mode, p, cfg, got, want)


def test_tables_end_inside_the_graph(gat, orc, gpu):
    """20,000 vertices: the tables cover the first 16,384, and 4,096 tables of
    a pool are shared by all the keys."""
    g = gat.Graph.chung_lu(20000, 4.0, 2.1, 40, 7)
    off, adj = g.csr()
    for p in (C5, HOUSE, cycle(4)):
        plan = gat.Plan(g, [p], "unique")
        want = [orc.unique_count(off, adj, p)]
        for cfg in ({}, {"split_us": 1}, {"hub_degree": 16}):
            assert plan.count(cfg)[0] == want, (p, cfg)


def test_epochs_and_replays(gat, orc, gpu, graphs):
    """More counts than there are epochs, with replays and accounted counts
    (which use no tables) between them, and shards of different roots."""
    g = graphs["rmat8"]
    off, adj = g.csr()
    plan = gat.Plan(g, [C5, HOUSE], "unique")
    want = [orc.unique_count(off, adj, p) for p in (C5, HOUSE)]
    n = g.v_cnt()
    for i in range(270):
        assert plan.count()[0] == want, i
        if i % 60 == 0:
            assert plan.count(graph_replays=3)[0] == want
            assert plan.count(account=True)[0] == want
            parts = [plan.count_shard(a, b)[0] for a, b in ((0, 5), (5, n // 2), (n // 2, n))]
            div = [plan.count_info(k)["divisor"] for k in (0, 1)]
            assert [sum(x) // d for x, d in zip(zip(*parts), div)] == want
