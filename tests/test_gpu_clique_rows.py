"""Rows and counts of the bitmap clique store at the edges of its tiers (GPU).
Closed forms: in a circulant graph (each vertex joined to its k nearest ids on
both sides of a ring of n > 3 k) every vertex but the last k has d = k
neighbours below it and there are n C(k, j-1) j-cliques; on the complete graph
K_m d takes every value up to m - 1 and there are C(m, j). The oracle gives
the accounted bytes and the counts of random graphs."""
import math

import numpy as np
import pytest

from patterns import clique

pytestmark = pytest.mark.gpu


def circulant(gat, n, k):
    v = np.repeat(np.arange(n, dtype=np.int64), k)
    step = np.tile(np.arange(1, k + 1, dtype=np.int64), n)
    return gat.Graph.from_edges(n, v, (v + step) % n)


def complete(gat, m):
    i, j = np.triu_indices(m, 1)
    return gat.Graph.from_edges(m, i, j)


# d = 2 and 11 take one pair per lane, 12 to 64 one wave, 65 a workgroup; with
# 40,000 vertices the core bitmap ends inside the graph (from 11,585 vertices
# on at k = 2 to 36,500 at k = 65), so both ways to build a row run
@pytest.mark.parametrize("k", [2, 3, 8, 11, 12, 32, 33, 63, 64, 65])
def test_circulant(gat, gpu, k):
    n = 40000
    g = circulant(gat, n, k)
    top = 6 if k <= 33 else 5
    for kmax in (3, top):
        js = list(range(3, kmax + 1))
        want = [n * math.comb(k, j - 1) for j in js]
        for cfg in ({}, {"queue_chunk": 1, "waves_per_cu": 2}, {"queue_chunk": 100, "slot_capacity": 32}):
            got, _ = gat.Plan(g, [clique(j) for j in js], "unique").count(cfg)
            assert got == want, (k, kmax, cfg, got, want)


# the last vertices of each LDS tier (256, 512, 1,024) and the first of the next
@pytest.mark.parametrize("m,ks", [(66, (3, 4, 5, 6)), (130, (4, 5, 6)), (258, (3, 4, 5)), (514, (4, 5)),
                                  (1030, (3, 4))])
def test_complete_graph_tier_edges(gat, gpu, m, ks):
    got, _ = gat.Plan(complete(gat, m), [clique(k) for k in ks], "unique").count()
    assert got == [math.comb(m, k) for k in ks]


def test_complete_graph_k5_widest_rows(gat, gpu):
    m = 1025  # d = 1,024: every tile of the widest LDS rows is full
    got, _ = gat.Plan(complete(gat, m), [clique(5)], "unique").count()
    assert got == [math.comb(m, 5)]


@pytest.mark.parametrize("n,p,cap", [(90, 0.7, 32), (150, 0.5, 64), (150, 0.5, 32)])
def test_random_tiers_counts_and_walg(gat, orc, gpu, n, p, cap):
    """Dense random graphs whose vertices take the workgroup tier: counts and
    W_alg of the oracle, whole and over a partition of the roots."""
    g = gat.Graph.erdos_renyi(n, p, 5)
    ro, ra = orc.relabel(*g.csr())
    for kmax in (4, 5):
        want_c, want_w = orc.clique_bitmap_walg(ro, ra, kmax)
        plan = gat.Plan(g, [clique(k) for k in range(3, kmax + 1)], "unique")
        got, st = plan.count({"slot_capacity": cap}, account=True)
        assert got[-1] == want_c and st["alg_bytes"] == want_w, (kmax, got, want_c, st["alg_bytes"], want_w)
        parts = [plan.count_shard(a, b, {"slot_capacity": cap})[0] for a, b in ((0, 7), (7, n - 3), (n - 3, n))]
        assert [sum(x) for x in zip(*parts)] == got


def test_replays_and_batches_agree(gat, gpu):
    """Captured replays of a batched plan that reaches three tiers, with eager
    counts between them."""
    g = gat.Graph.rmat(13, 32, 0.57, 0.19, 0.19, 3)
    plan = gat.Plan(g, [clique(3), clique(4), clique(5)], "unique")
    want, _ = plan.count({"slot_capacity": 32})
    single = [gat.Plan(g, [clique(k)], "unique").count()[0][0] for k in (3, 4, 5)]
    assert want == single
    for _ in range(3):
        assert plan.count(graph_replays=3)[0] == want
        assert plan.count()[0] == want
