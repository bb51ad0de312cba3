"""Runs a test's code in a child process whose HIP runtime is fake_hip.cpp:
the host code's allocations, uploads, launches and events without a GPU."""
import json
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
PRELUDE = """
import ctypes as C, json, sys, threading, time
fake = C.CDLL(%r, mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_char_p
fake.fake_live.restype = C.c_size_t
fake.fake_limit.argtypes = [C.c_size_t]
fake.fake_refuse.argtypes = [C.c_size_t, C.c_int]
sys.path[:0] = [%r, %r]
import graphautotune_amd as gat
from graphautotune_amd._lib import GatError
from patterns import C5, HOUSE, K4, TRIANGLE, clique
def calls(word=""):  # the recorded calls that begin with word
    return [l for l in fake.fake_log().decode().splitlines() if l.startswith(word)]
def result(x):
    print("RESULT " + json.dumps(x), flush=True)
"""


def build(folder):
    lib = os.path.join(str(folder), "fake_hip.so")
    cxx = os.environ.get("CXX", "g++")
    r = subprocess.run([cxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                        os.path.join(HERE, "fake_hip.cpp"), "-o", lib, "-lpthread"], text=True, stdout=subprocess.PIPE,
                       stderr=subprocess.STDOUT)
    assert r.returncode == 0, r.stdout
    return lib


def run(lib, code, timeout=100):
    r = subprocess.run([sys.executable, "-c", PRELUDE % (lib, ROOT, HERE) + code], text=True, timeout=timeout, cwd=ROOT,
                       stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    lines = [l for l in r.stdout.splitlines() if l.startswith("RESULT ")]
    assert r.returncode == 0 and len(lines) == 1, r.stdout
    return json.loads(lines[0][7:])
