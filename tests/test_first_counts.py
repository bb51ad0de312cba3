"""First counts of several plans of one graph on several threads share one
device copy of it, with a runtime that records its calls and no GPU."""
import pytest

import fakehip


@pytest.mark.parametrize("pattern", ["HOUSE", "K4"])  # array store, clique store
def test_one_upload(tmp_path, pattern):
    uploads = fakehip.run(fakehip.build(tmp_path), """
g = gat.Graph.rmat(10, 16, .57, .19, .19, 1)
plans = [gat.Plan(g, [%s], "unique") for _ in range(4)]
fake.fake_slow_copies(50)
threads = [threading.Thread(target=p.count) for p in plans]
for t in threads:
    t.start()
for t in threads:
    t.join()
result(len(calls("copy %%d" %% (4 * g.e_cnt()))))
""" % pattern)
    assert uploads == 1
