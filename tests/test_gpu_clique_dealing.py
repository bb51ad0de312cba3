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
