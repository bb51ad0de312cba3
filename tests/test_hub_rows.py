"""Hub bitmaps as the host code keeps them, with a runtime that records its
calls and no GPU: plans of different thresholds share one set of rows, a set in
use is not freed, and a set that could not be built is built by the next count."""
import pytest

import fakehip

HUB = "launch _ZN4gatk15hub_rows_kernel"


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return fakehip.build(tmp_path_factory.mktemp("fake"))


@pytest.mark.parametrize("mode", ["unique", "reference"])  # degree order, and rows found through a map
def test_thresholds_share_one_set(fake, mode):
    """The default takes vertices below degree 256 too; counts with the
    threshold 256 of gat_default_config between them do not build it anew."""
    builds = fakehip.run(fake, """
g = gat.Graph.rmat(10, 16, .57, .19, .19, 1)
plans = [gat.Plan(g, [HOUSE], %r) for _ in range(2)]
built = []
for cfg in ({"hub_degree": 100000}, {}, {"hub_degree": 256}, {}, gat.core.default_config(), {"hub_degree": 100000}, {}, {"hub_degree": 1},
            {"hub_degree": 1}, {}, {"hub_degree": -1}):
    calls()
    plans[len(built) %% 2].count(cfg)
    built.append(len(calls(%r)))
result(built)
""" % (mode, HUB))
    assert builds == [0, 1, 0, 0, 0, 0, 0, 1, 0, 0, 0]


@pytest.mark.parametrize("refused", [12500, 400000])
def test_failed_build_is_repeated(fake, refused):
    """Rows are 12,500 bytes each here, for a few vertices, and the map from
    vertices to rows 400,000: without memory for one of them the count fails,
    and the next one builds what it needs."""
    first, builds = fakehip.run(fake, """
g = gat.Graph.erdos_renyi(100000, 4 / 100000, 1)
p = gat.Plan(g, [HOUSE], "reference")
p.count({"hub_degree": -1})  # everything but the bitmaps
fake.fake_refuse(%d, -1)
try:
    p.count({"hub_degree": 14})
    first = "counted"
except GatError:
    first = "refused"
fake.fake_refuse(1 << 60, 0)
calls()
p.count({"hub_degree": 14})
result([first, len(calls(%r))])
""" % (refused, HUB))
    assert first == "refused" and builds == 1


def test_rows_in_use_are_not_freed(fake):
    """While one plan's count is under way, another plan of the graph needs
    more rows: the old ones stay until the first count is done."""
    during, after = fakehip.run(fake, """
g = gat.Graph.rmat(10, 16, .57, .19, .19, 1)
a, b = (gat.Plan(g, [HOUSE], "unique") for _ in range(2))
b.count({"hub_degree": -1})
calls()
a.count({"hub_degree": 200})
off = g.csr()[0]
rows = 128 * sum(off[v + 1] - off[v] >= 200 for v in range(1024))
assert "malloc %d" % rows in calls("malloc")
fake.fake_hold()
t = threading.Thread(target=lambda: a.count({"hub_degree": 200}))
t.start()
while not fake.fake_held():
    time.sleep(0.01)
calls()
b.count({"hub_degree": 2})
freed = "free %d" % rows
during = freed in calls("free")
fake.fake_release()
t.join()
result([during, freed in calls("free")])
""")
    assert not during and after
