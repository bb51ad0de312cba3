"""How the clique store deals out vertices (GPU): on a graph without heavy
vertices every wave of the main launch takes its share and no more, whatever
queue_chunk says; a tier with many light items counts each of them once."""
import math

import numpy as np
import pytest

from patterns import clique

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("config", [{}, {"queue_chunk": 4, "block_waves": 2}, {"queue_chunk": 1}])
def test_waves_take_equal_shares(gat, gpu, config):
    n = 50000
    g = gat.Graph.erdos_renyi(n, 40 / n, 1)
    got, st = gat.Plan(g, [clique(3)], "unique").count(config, timeline=True)
    assert got == [g.triangles()]
    main = st["timeline"][st["timeline"][:, 0] == 0]
    assert main[:, 6].max() <= math.ceil(n / len(main)), (len(main), main[:, 6].max())


def circulant(gat, n, k):
    v = np.repeat(np.arange(n, dtype=np.int64), k)
    step = np.tile(np.arange(1, k + 1, dtype=np.int64), n)
    return gat.Graph.from_edges(n, v, (v + step) % n)


# tier 0 has 39,930 and 1,930 vertices: several per grab of its queue, and one;
# tier 1 by itself. Beside the closed form, sparse rows: no pair in most of them
@pytest.mark.parametrize("n,k", [(40000, 70), (2000, 70), (3000, 300)])
def test_tier_items(gat, gpu, n, k):
    got, _ = gat.Plan(circulant(gat, n, k), [clique(j) for j in (3, 4, 5)], "unique").count()
    assert got == [n * math.comb(k, j - 1) for j in (3, 4, 5)]


def test_tiers_of_a_sparse_graph(gat, gpu):
    """Rows almost without bits: triangles from the host, other cliques against
    the array store."""
    g = gat.Graph.erdos_renyi(30000, 200 / 30000, 7)
    plan = gat.Plan(g, [clique(3), clique(4), clique(5)], "unique")
    got, _ = plan.count()
    assert got[0] == g.triangles() and got == plan.count({"vertex_store": 1})[0]


def test_k6_sparse_vertices_stay_in_the_main_launch(gat, gpu):
    """No vertex has 65 neighbours below it, hundreds have more than 32, and
    hardly any pair of those is adjacent: nothing is left to the tiers."""
    g = gat.Graph.erdos_renyi(50000, 40 / 50000, 1)
    plan = gat.Plan(g, [clique(3), clique(6)], "unique")
    got, st = plan.count({"slot_capacity": 64}, timeline=True)
    tiers = st["timeline"][st["timeline"][:, 0] > 0]
    assert st["overflow_tasks"] == 0 and tiers[:, 6].sum() == 0
    assert got == [g.triangles(), 0]


@pytest.mark.parametrize("k", [32, 33, 48, 63, 64, 65])
def test_k6_dense_vertices_go_to_the_tier(gat, gpu, k):
    n = 3000
    for ks in ((6,), (3, 4, 5, 6)):
        plan = gat.Plan(circulant(gat, n, k), [clique(j) for j in ks], "unique")
        for _ in range(2):
            got, st = plan.count(timeline=True)
            assert got == [n * math.comb(k, j - 1) for j in ks]
            tiers = st["timeline"][st["timeline"][:, 0] > 0]
            assert tiers[:, 6].sum() >= (n - k) * (k > 32)
        parts = [plan.count_shard(a, b)[0] for a, b in ((0, 40), (40, n - 7), (n - 7, n))]
        assert [sum(x) for x in zip(*parts)] == got
        assert plan.count(graph_replays=3)[0] == got


@pytest.mark.parametrize("p", [0.3, 0.5, 0.7])  # around a quarter of the pairs adjacent
def test_k6_walg_is_charged_once(gat, orc, gpu, p):
    g = gat.Graph.erdos_renyi(100, p, 5)
    ro, ra = orc.relabel(*g.csr())
    want_c, want_w = orc.clique_bitmap_walg(ro, ra, 6)
    got, st = gat.Plan(g, [clique(6)], "unique").count(account=True)
    assert got == [want_c] and st["alg_bytes"] == want_w
