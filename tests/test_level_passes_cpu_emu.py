"""One-pass level kernels and the single-workgroup cycle on the CPU (no GPU).

The march over a multigrid level (nyl_march.hip) and the cycle of the small
levels (nyl_cycle.hip) must give the same bits as the per-cell kernels they
stand for, for partial tiles, every periodicity and one-cell axes; the
device-side stop rule must take the host loop's decisions.  The kernel sources
are built for the host as in test_kernels_cpu_emu.py, with AddressSanitizer.
"""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
EMU = os.path.join(HERE, "cpu_emu")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")


@pytest.mark.parametrize("name", ["march_emu", "cycle_emu"])
def test_level_passes_match_per_cell_forms_bitwise(name, tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ is not available")
    exe = str(tmp_path / name)
    src = os.path.join(EMU, name + ".cpp")
    build = [gxx, "-std=c++17", "-O1", "-fsanitize=address", "-fno-omit-frame-pointer",
             "-I", EMU, "-I", INCLUDE, src, "-lpthread", "-o", exe]
    subprocess.run(build, check=True, timeout=900)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=900)
    tail = r.stdout[-3000:] + r.stderr[-3000:]
    assert r.returncode == 0 and "ALL OK" in r.stdout, tail
