"""Roofline entries of the bench's auxiliary lines, from made-up figures."""
import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)


@pytest.mark.parametrize("traffic,frac", [(4.0e10, 0.5), (None, None)])
def test_iep_fraction_is_of_measured_traffic(traffic, frac):
    """W_alg of the accounted pass is 600 times what a count with kept values
    moves: no fraction of the memory's peak."""
    import bench
    r = bench.iep_roofline("gatk::engine_kernel<false>", 10.0, 600 * 4.0e10, traffic)
    assert r["frac"] == (pytest.approx(frac) if frac else None) and r["bound"] == "hbm"
    assert r["achieved"] == (pytest.approx(4000.0) if traffic else None)
    assert r["work_equivalent_gbps"] == pytest.approx(600 * 4000.0)


def test_clique_groups_show_every_kernel():
    import bench
    group = "tiers 0 and 1"
    names = bench.CLIQUE_GROUPS[group]
    prof = {"derived": {n: {"valu_issue": 0.1 * (i + 1)} for i, n in enumerate(names)}}
    r = bench.clique_roofline(group, 10.0, 4.0e12, prof)
    assert {r["counters_kernel"], *r["counters_others"]} == set(names)
    assert r["counters"]["valu_issue"] == pytest.approx(0.1) and len(names) == 2
