"""Workgroup barriers in the kernels' sources: every wave of a workgroup has to
reach one, so none may stand behind a return that only some of the waves take."""
import glob
import os
import re

import pytest

from conftest import ROOT

HIP = os.path.join(ROOT, "biobench2_amd", "csrc", "hip")
BARRIER = re.compile(r"__syncthreads|lds_barrier\(\)|s_barrier|stage_table\(")
# a return that depends on the wave's number
LEAVES = re.compile(r"if \([^;{}]*(\bwv\b|threadIdx\.x >> 6)[^;{}]*\) return;")


def kernels(path):
    src = re.sub(r"//[^\n]*", "", open(path).read())
    for m in re.finditer(r"__global__[^;{]*?\b(k_\w+)\s*\(", src):
        at = src.index("{", src.index(")\n", m.end()))
        depth, i = 0, at
        while True:
            depth += {"{": 1, "}": -1}.get(src[i], 0)
            i += 1
            if depth == 0:
                break
        yield m.group(1), src[at:i]


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(HIP, "*.hip"))), ids=os.path.basename)
def test_no_barrier_behind_a_return_of_some_waves(path):
    found = dict(kernels(path))
    assert os.path.basename(path) == "p7g_runtime.hip" or found
    for name, body in found.items():
        left = LEAVES.search(body)
        if left:
            late = BARRIER.search(body, left.end())
            assert not late, (name, left.group(0), late.group(0))
