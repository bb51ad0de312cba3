"""What the times of a count cover, on a runtime that records its calls and no
GPU: `seconds` starts before the tables of kept counts are cleared, and
`main_kernel_ms` after that."""
import pytest

import fakehip


# house clears edge tables in every count; C5 its pool in the first of 254
@pytest.mark.parametrize("pattern,counts,clears", [("HOUSE", 2, 2), ("C5", 1, 1), ("C5", 2, 0), ("K4", 2, 0)])
def test_clearing_is_part_of_the_time(tmp_path, pattern, counts, clears):
    log = fakehip.run(fakehip.build(tmp_path), """
p = gat.Plan(gat.Graph.rmat(10, 16, .57, .19, .19, 1), [%s], "unique")
for _ in range(%d):
    calls()
    p.count()
result(calls())
""" % (pattern, counts))
    fills = [i for i, l in enumerate(log) if "fill_u64" in l and not any("hub_rows" in x for x in log[i:i + 2])]
    events = [(i, l.split()[1]) for i, l in enumerate(log) if l.startswith("event")]
    spans = [l.split()[1:] for l in log if l.startswith("elapsed")]
    whole, main = spans[0], spans[1]
    at = {e: i for i, e in events}
    # the control words are cleared before the count starts, the tables after it
    tables = [i for i in fills if i > at[whole[0]]]
    assert len(fills) - len(tables) == 1 and len(tables) >= clears and bool(tables) == bool(clears)
    assert all(at[whole[0]] < i < at[main[0]] for i in tables)
    assert at[main[0]] < at[main[1]] and (tables or main[0] == whole[0])
