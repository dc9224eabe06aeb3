"""The buffer offsets of the attention mass chain (cuda_inf_amd/csrc/h2o_chain.h)
stay inside the chunk or are refused, whichever way the hardware's range check
takes a scalar offset; with the step's row in the scalar offset they would not."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_chain_loads_in_bounds(tmp_path):
    exe = str(tmp_path / "h2o_chain_check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(HERE, "..", "cuda_inf_amd", "csrc"),
                    os.path.join(HERE, "h2o_chain_check.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    r = subprocess.run([exe, "scalar"], capture_output=True, text=True, timeout=60)
    assert r.returncode == 1, "rows in the scalar offset went unnoticed"
