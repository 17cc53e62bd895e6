"""What the library's host code plans, checked on the CPU (no GPU): the host
code is built with g++ against a stand-in of the HIP runtime in which memory
is host memory and a launch runs nothing (tests/cpu_emu/host)."""
import concurrent.futures
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HOST = os.path.join(HERE, "cpu_emu", "host")
CSRC = os.path.join(ROOT, "nyles_amd", "csrc")


def build(tmp_path, name, without=()):
    """tests/cpu_emu/host/<name>.cpp with the library's sources that it does not
    include itself"""
    from nyles_amd.build import SOURCES
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    flags = ["-std=c++17", "-O1", "-w", "-I", HOST, "-I", os.path.join(HERE, "cpu_emu"),
             "-I", os.path.join(ROOT, "include")]
    srcs = [os.path.join(CSRC, s) for s in SOURCES
            if s not in without and s not in ("nyl_noalloc.hip", "nyl_mgfor.hip")]
    srcs += [os.path.join(HOST, "emu_host.cpp"), os.path.join(HOST, name + ".cpp")]
    objs = [str(tmp_path / (os.path.basename(s) + ".o")) for s in srcs]
    with concurrent.futures.ThreadPoolExecutor(max_workers=4) as ex:
        list(ex.map(lambda so: subprocess.run(
            [gxx] + flags + ["-x", "c++", "-c", so[0], "-o", so[1]], check=True, timeout=600),
            zip(srcs, objs)))
    exe = str(tmp_path / name)
    subprocess.run([gxx] + objs + ["-lpthread", "-o", exe], check=True, timeout=600)
    return exe


def run(exe):
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600)
    tail = r.stdout[-3000:] + r.stderr[-3000:]
    assert r.returncode == 0 and "ALL OK" in r.stdout, tail


def test_batch_block_sums_stay_inside_their_partials(tmp_path):
    run(build(tmp_path, "batch_plan", without=("nyl_batch.hip",)))


def test_stage_grids_stay_within_the_limits(tmp_path):
    run(build(tmp_path, "stage_grids", without=("nyl_api.hip",)))
