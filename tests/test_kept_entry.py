"""Entries of the tables of kept counts: tag, value and epoch come from one
8-byte access however the code around it uses them. The probe kernels are
compiled for gfx950 and their assembly read; a plain load of the same pair
whose halves are used in different branches is two 4-byte loads there."""
import os
import re
import subprocess

import pytest

from graphautotune_amd import build

PROBE = r"""
#include "kept.h"
using gatk::KeptEntry;
extern "C" __global__ void halves_apart(const KeptEntry *t, const int *at, unsigned tag, unsigned epoch, int *out) {
    const KeptEntry::Read e = t[at[threadIdx.x]].read();
    if (e.tag != tag) return;
    out[threadIdx.x] = e.serves(tag, epoch) ? e.value() : -1;
}
extern "C" __global__ void tag_alone(const KeptEntry *t, const int *at, unsigned tag, int *out) {
    out[threadIdx.x] = t[at[threadIdx.x]].read().tag == tag;
}
extern "C" __global__ void put(KeptEntry *t, const int *at, unsigned tag, const int *value, unsigned epoch) {
    t[at[threadIdx.x]].write(tag, value[threadIdx.x], epoch);
}
"""


def compile_probe(tmp_path, source, *args):
    src = tmp_path / "probe.hip"
    src.write_text(source)
    flags = [f for f in build.HIP_FLAGS if f != "-fPIC"]
    return subprocess.run([build.HIPCC, *flags, "--cuda-device-only", *args, str(src)], text=True,
                          stdout=subprocess.PIPE, stderr=subprocess.STDOUT)


@pytest.fixture(scope="module")
def assembly(tmp_path_factory):
    d = tmp_path_factory.mktemp("kept")
    out = d / "probe.s"
    r = compile_probe(d, PROBE, "-S", "-o", str(out))
    assert r.returncode == 0, r.stdout
    text = out.read_text()
    return {k: re.search(r"^%s:(.*?)s_endpgm" % k, text, re.S | re.M).group(1)
            for k in ("halves_apart", "tag_alone", "put")}


@pytest.mark.parametrize("kernel", ["halves_apart", "tag_alone"])
def test_read_is_one_access(assembly, kernel):
    # beside the entry, each kernel loads its index (4 bytes)
    loads = re.findall(r"(?:global|flat)_load_\w+", assembly[kernel])
    assert sorted(loads) == ["global_load_dword", "global_load_dwordx2"], loads


def test_write_is_one_access(assembly):
    stores = re.findall(r"(?:global|flat)_store_\w+", assembly["put"])
    assert stores == ["global_store_dwordx2"], stores


@pytest.mark.parametrize("use", ["int x = (int)t->word;", "t->word = 1;", "KeptEntry e = *t; int x = (int)e.word;"])
def test_no_other_access_compiles(tmp_path, use):
    r = compile_probe(tmp_path, PROBE + "__global__ void other(KeptEntry *t) { %s }" % use, "-fsyntax-only")
    assert r.returncode != 0 and "private" in r.stdout, r.stdout


def test_engine_holds_entries_only():
    src = open(os.path.join(build.CSRC, "engine.hip")).read()
    assert "KeptEntry *pool;" in src and "uint2" not in src
