"""The row count that a packed pass's GEMM tiles are chosen for: the live share
of the last batch, and of the last single sequence, on the stream. The check is
compiled from the library's own header as host code
(tests/cpu_checks/tile_hint.cpp)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="needs hipcc for the HIP headers")
def test_tile_hint(tmp_path):
    exe = tmp_path / "tile_hint"
    subprocess.run([HIPCC, "-O1", "-std=c++17",
                    "-I", os.path.join(ROOT, "npu-embeddings-xdna1_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"),
                    "-o", str(exe), os.path.join(HERE, "cpu_checks", "tile_hint.cpp")],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.strip() == "ok"
