"""Buffers that are kept between calls (single targets' residues, rows and pinned
memory), grown by keep_at_least: after an allocation that failed, the next call
that needs less must not take the old capacity for the buffer that is gone.
Host code, compiled with an allocator that fails on request."""
import os
import subprocess

from conftest import ROOT


def test_failed_growth_leaves_no_capacity(tmp_path):
    exe = str(tmp_path / "keep")
    host = os.path.join(ROOT, "biobench2_amd", "csrc", "host")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-I", host, "-o", exe,
                    os.path.join(ROOT, "tests", "abi", "keep_buffer.cpp")], check=True)
    # status, capacity, buffer there, buffers alive, allocations so far
    run = subprocess.run([exe, "10", "5", "-100", "5", "5", "20", "-30", "-25", "1"], capture_output=True, text=True, check=True)
    got = [tuple(map(int, line.split())) for line in run.stdout.split("\n") if line]
    assert got == [(0, 10, 1, 1, 1), (0, 10, 1, 1, 1),      # made, and kept for less
                   (2, 0, 0, 0, 2),                          # growth failed: nothing is held
                   (0, 5, 1, 1, 3), (0, 5, 1, 1, 3),         # a smaller call allocates again
                   (0, 20, 1, 1, 4), (2, 0, 0, 0, 5), (2, 0, 0, 0, 6), (0, 1, 1, 1, 7)]


def test_every_kept_buffer_of_single_targets_grows_so():
    src = open(os.path.join(ROOT, "biobench2_amd", "csrc", "hip", "p7g_runtime.hip")).read()
    one = src[src.index("struct Single {"):src.index("p7_gpu_ForwardParser(")]
    for field, cap in (("res", "cap"), ("xmx", "xcap"), ("pin", "pcap")):
        assert f"keep_at_least(o.{field}, o.{cap}," in one, field
    batch = src[src.index("\nbatch_reserve("):]
    batch = batch[:batch.index("hipMalloc")]
    assert "b.nprof_cap = 0" in batch and "b.n_cap = 0" in batch and "b.mask_cap = 0" in batch
