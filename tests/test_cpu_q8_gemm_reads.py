"""CPU: every load of the batched Q8_0 GEMM's kernels lies inside its matrix or workspace.

The kernels load a few chunks ahead, past the end of a row; on a GPU the values read there
are never used, so no result can show where they came from. Their offsets are plain integer
functions (ferrum_amd/csrc/fkv_gemm_at.h), walked here for every lane, wave and chunk."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_every_load_is_inside_its_matrix_or_workspace(tmp_path):
    exe = tmp_path / "gemm_at_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-o", str(exe),
                    os.path.join(HERE, "gemm", "gemm_at_check.cpp")], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.stdout.strip() == "ok", out.stdout
    assert out.returncode == 0
