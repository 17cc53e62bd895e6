"""The stage kernel with 16 bytes of cells per thread, and the FP64
reconstruction with its short division, on the CPU (no GPU): the same bits as
the per-cell kernel and as the reference's expression.  Built for the host as
in test_kernels_cpu_emu.py, with AddressSanitizer."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "cpu_emu")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")


def test_stage_forms_match_per_cell_form_bitwise(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path / "stage_flat_emu")
    src = os.path.join(EMU, "stage_flat_emu.cpp")
    build = [gxx, "-std=c++17", "-O1", "-fsanitize=address", "-fno-omit-frame-pointer",
             "-I", EMU, "-I", INCLUDE, src, "-lpthread", "-o", exe]
    subprocess.run(build, check=True, timeout=900)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=900)
    tail = r.stdout[-3000:] + r.stderr[-3000:]
    assert r.returncode == 0 and "ALL OK" in r.stdout, tail
