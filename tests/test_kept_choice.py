"""Which leaf counts are kept in tables on which graph, from the kernels and
allocations of a count on a runtime that records its calls and has no GPU: where a
value is hardly asked for again, the walk without tables runs and nothing is
allocated for them."""
import pytest

import fakehip

PLAIN, KEPT, PAIR = "engine_plain_kernel", "engine_kernel", "engine_pair_kernel"


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fakehip.build(tmp_path_factory.mktemp("fake"))


# degree 8: no value is wanted often enough, but the pair sweep pays for itself;
# degree 24: edges (whole lists) only; R-MAT: all
@pytest.mark.parametrize("graph,pattern,mode,kernel,edges,pools", [
    ("erdos_renyi(20000, 8 / 20000, 1)", "HOUSE", "unique", PLAIN, 0, 0),
    ("erdos_renyi(20000, 8 / 20000, 1)", "C5", "reference", PLAIN, 0, 0),
    ("erdos_renyi(20000, 8 / 20000, 1)", "C5", "unique", PAIR, 0, 1),
    ("erdos_renyi(20000, 24 / 20000, 1)", "HOUSE", "unique", KEPT, 1, 0),
    ("rmat(10, 16, .57, .19, .19, 1)", "HOUSE", "unique", KEPT, 2, 1),
    ("rmat(10, 16, .57, .19, .19, 1)", "C5", "reference", KEPT, 0, 1),
])
def test_choice(fake, graph, pattern, mode, kernel, edges, pools):
    got = fakehip.run(fake, """
g = gat.Graph.%s
gat.Plan(g, [TRIANGLE], %r).count({"vertex_store": 1, "split_us": -1})  # the graph is on the device
p = gat.Plan(g, [%s], %r)
calls()
p.count({"split_us": -1, "hub_degree": -1})
l = calls()
sizes = [int(x[7:]) for x in l if x.startswith("malloc")]
edge, overflow = 4 * g.e_cnt(), 8 * (g.e_cnt() + 1)  # the pool, if any, comes after these
result([[x for x in ("engine_plain_kernel", "engine_kernel", "engine_pair_kernel") if any("%%d%%sILb0E" %% (len(x), x) in y for y in l)],
        sizes.count(edge), int(sizes[-1] not in (edge, overflow))])
""" % (graph, mode, pattern, mode))
    assert got == [[kernel], edges, pools]
