"""Counts with less of the memory that they can do without, or none (GPU): the
allocation is refused in a child process, whose counts are compared with those
of this one."""
import json
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu
HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

CHILD = """
import ctypes as C, json, sys
limit = C.CDLL(%r, mode=C.RTLD_GLOBAL)
limit.limit_refuse.argtypes = [C.c_size_t, C.c_size_t]
sys.path[:0] = [%r, %r]
import graphautotune_amd as gat
from patterns import C5, HOUSE, K4, clique
g = gat.Graph.rmat(12, 12, .57, .19, .19, 5)
gat.Plan(g, [HOUSE], "unique").count_shard(0, 1, {"hub_degree": -1, "split_us": -1})  # the graph is on the device
for sizes in %r:
    limit.limit_refuse(*sizes)
out = []
for patterns, mode, config in %r:
    plan = gat.Plan(g, patterns, mode)
    out.append([plan.count(config)[0], plan.count(config)[0], plan.count(config, graph_replays=2)[0]])
print("RESULT " + json.dumps([limit.limit_refused(), out]), flush=True)
"""


@pytest.fixture(scope="module")
def limiter(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("limit") / "malloc_limit.so")
    r = subprocess.run([os.environ.get("CXX", "g++"), "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__",
                        "-I/opt/rocm/include", os.path.join(HERE, "malloc_limit.cpp"), "-o", lib, "-ldl"], text=True,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    assert r.returncode == 0, r.stdout
    return lib


MB = 1 << 20


def sizes(*mb):  # of pools: a budget in MiB, less up to three tables
    return [(x * MB - 3 * 8 * 4096, x * MB + 1) for x in mb]


# 4,096 vertices: pools of 128 MiB (keyed by a vertex) or 512 MiB (by an edge),
# 512 bytes a hub row, 888 vertices of degree >= 16, and 264,064 words of core rows
@pytest.mark.parametrize("refused", [sizes(512, 128), sizes(512, 128, 32, 8), [(888 * 512, 888 * 512 + 1)],
                                     [(4 * 264064, 4 * 264064 + 1)]],
                         ids=["smaller pools", "no tables", "hub rows from 256 on", "no core bitmap"])
def test_counts_are_the_same(gat, gpu, limiter, refused):
    from patterns import C5, HOUSE, K4, clique, connected_patterns
    plans = [([C5], "unique", {}), ([HOUSE], "unique", {"split_us": 1}), ([C5], "reference", {}),
             (connected_patterns(5)[:8], "unique", {}), ([clique(3), K4, clique(5)], "unique", {}),
             ([clique(6)], "unique", {"slot_capacity": 32})]
    g = gat.Graph.rmat(12, 12, 0.57, 0.19, 0.19, 5)
    want = [gat.Plan(g, p, m).count(c)[0] for p, m, c in plans]
    r = subprocess.run([sys.executable, "-c", CHILD % (limiter, ROOT, HERE, refused, plans)], text=True, timeout=100,
                       cwd=ROOT, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    line = [l for l in r.stdout.splitlines() if l.startswith("RESULT ")]
    assert r.returncode == 0 and len(line) == 1, r.stdout
    times, got = json.loads(line[0][7:])
    assert times > 0
    assert got == [[w, w, w] for w in want]
