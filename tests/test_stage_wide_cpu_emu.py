"""The stage and tracer kernels of wide planes, and the short FP64 division of
the reconstructions over the whole range it is used on, on the CPU (no GPU),
built for the host as in test_kernels_cpu_emu.py, with AddressSanitizer."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "cpu_emu")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")


@pytest.mark.parametrize("name", ["stage_wide_emu", "division_emu"])
def test_wide_stage_forms_bitwise(name, tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path / name)
    build = [gxx, "-std=c++17", "-O1", "-fsanitize=address", "-fno-omit-frame-pointer",
             "-I", EMU, "-I", INCLUDE, os.path.join(EMU, name + ".cpp"), "-lpthread",
             "-o", exe]
    subprocess.run(build, check=True, timeout=900)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=900)
    tail = r.stdout[-3000:] + r.stderr[-3000:]
    assert r.returncode == 0 and "ALL OK" in r.stdout, tail
