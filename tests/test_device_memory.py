"""Device memory that counts can do without (tables of kept counts, bitmaps), on
a runtime that records its calls and refuses allocations, and without a GPU: it
is given back where a count cannot go on otherwise, never while a count uses
it, and counts go on with less of it or none."""
import pytest

import fakehip

PLAIN, PAIR = "launch _ZN4gatk19engine_plain_kernel", "launch _ZN4gatk18engine_pair_kernel"


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fakehip.build(tmp_path_factory.mktemp("fake"))


PLANS = """
g = gat.Graph.rmat(10, 16, .57, .19, .19, 1)
cfg = {"split_us": -1}
def plan():
    return gat.Plan(g, [HOUSE], "unique")
first = plan()
first.count(cfg)
second = plan()
calls()
second.count(cfg)
sizes = [int(l.split()[1]) for l in calls("malloc")]
tables = [s for s in sizes if s in (4 * g.e_cnt(), 8 << 20)]  # two edge tables, a pool of 1,024 tables
assert len(tables) == 3
needed = sum(sizes) - sum(tables)
"""


def test_idle_plans_give_their_tables_back(fake):
    """Room for what twenty more plans cannot do without, and not for tables."""
    counted = fakehip.run(fake, PLANS + """
fake.fake_limit(fake.fake_live() + 20 * needed)
plans = [plan() for _ in range(20)]
for p in plans:
    p.count(cfg)
result(len(plans))
""")
    assert counted == 20


def test_tables_in_use_stay(fake):
    refused, during, after = fakehip.run(fake, PLANS + """
del second
third = plan()
fake.fake_limit(fake.fake_live() + needed - 1000)
fake.fake_hold()
t = threading.Thread(target=lambda: first.count(cfg))
t.start()
while not fake.fake_held():
    time.sleep(0.01)
calls()
refused = 0
try:
    third.count(cfg)
except GatError:
    refused = 1
pool = "free %d" % (8 << 20)
during = calls().count(pool)
fake.fake_release()
t.join()
calls()
third.count(cfg)
result([refused, during, calls().count(pool)])
""")
    assert (refused, during, after) == (1, 0, 1)


@pytest.mark.parametrize("plan,config", [("HOUSE", {"hub_degree": -1}), ("TRIANGLE", {"vertex_store": 1}), ("K4", {})])
def test_cost_model_takes_what_an_idle_plan_or_graph_holds(fake, plan, config):
    """Tables, hub bitmaps and the core bitmap, of 3 MB and more each."""
    ok = fakehip.run(fake, """
from graphautotune_amd.tuning.mlp import MLPCostModel
g = gat.Graph.rmat(13, 16, .57, .19, .19, 1)
p = gat.Plan(g, [%s], "unique")
p.count(%r)
fake.fake_limit(fake.fake_live())
m = MLPCostModel(96, 256)
fake.fake_limit(1 << 60)
p.count(%r)
result(m.n_params)
""" % (plan, config, config))
    assert ok == 96 * 256 + 256 + 256 * 256 + 256 + 256 + 1


def test_pool_shrinks_and_tables_are_left_out(fake):
    """20,000 vertices: a pool of 512 MiB, a quarter where that is refused, and
    none, with no edge tables held and no further requests for 64 counts."""
    got = fakehip.run(fake, """
g = gat.Graph.erdos_renyi(20000, 6 / 20000, 1)
cfg = {"split_us": -1}
def count(p):
    calls()
    p.count(cfg)
    l = calls()
    return {"refused": sum(x.startswith("refuse") for x in l), "plain": any(x.startswith(%r) for x in l),
            "pair": any(x.startswith(%r) for x in l), "pool": [int(x[7:]) for x in l if x.startswith("malloc")][-1]}
p = gat.Plan(g, [C5], "unique")
fake.fake_refuse(200 << 20, -1)
small = count(p)
p = gat.Plan(g, [C5], "unique")
fake.fake_refuse(8 << 20, -1)
none = count(p)
quiet = []
fake.fake_refuse(1 << 62, 0)
for _ in range(64):
    calls()
    p.count(cfg)
    l = calls()
    quiet.append(any(x.startswith("malloc") for x in l))
result([small, none, any(quiet), count(p)])
""" % (PLAIN, PAIR))
    small, none, asked, later = got
    assert small == {"refused": 1, "plain": False, "pair": True, "pool": 128 << 20}
    assert none["refused"] == 4 and none["plain"] and not none["pair"]
    assert not asked
    assert later["pair"] and later["pool"] == 512 << 20


def test_edge_tables_are_not_held_for_nothing(fake):
    """The pool is refused: what the edge tables took is free again."""
    got = fakehip.run(fake, """
g = gat.Graph.erdos_renyi(3000, 60 / 3000, 1)
gat.Plan(g, [TRIANGLE], "unique").count({"vertex_store": 1, "split_us": -1})  # the graph is on the device
p = gat.Plan(g, [HOUSE], "unique")
fake.fake_refuse(8000000, -1)  # pools have 8.4 MB and more, set buffers 4.7
calls()
p.count({"split_us": -1})
l = calls()
edges = " %d" % (4 * g.e_cnt())
result([l.count("malloc" + edges), l.count("free" + edges)])
""")
    assert got[0] > 0 and got[0] == got[1]


def test_cliques_without_a_core_bitmap(fake):
    launched = fakehip.run(fake, """
g = gat.Graph.rmat(10, 16, .57, .19, .19, 1)
gat.Plan(g, [HOUSE], "unique").count()   # the graph is on the device
p = gat.Plan(g, [K4], "unique")
fake.fake_refuse(67000, -1)              # 1,024 core rows take 67,456 bytes
calls()
p.count()
l = calls()
result([sum(x.startswith("refuse") for x in l), sum("clique_kernel" in x for x in l)])
""")
    assert launched[0] >= 1 and launched[1] == 1


@pytest.mark.parametrize("size", [8000, 10000, 1 << 20])  # the graph, the plan, its set buffers
def test_a_first_count_that_fails_can_be_repeated(fake, size):
    first = fakehip.run(fake, """
p = gat.Plan(gat.Graph.rmat(10, 16, .57, .19, .19, 1), [HOUSE], "unique")
fake.fake_refuse(%d, 1)
first = "counted"
try:
    p.count()
except GatError:
    first = "refused"
p.count()
result(first)
""" % size)
    assert first == "refused"
