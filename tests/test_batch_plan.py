"""The groups of a batch and their fuse limits
(hunyuansc25_amd/csrc/hgp_batchplan.hpp) on the host alone: built with g++
from tests/native/batch_plan_test.cpp and run."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_batch_plan(tmp_path):
    exe = str(tmp_path / "batch_plan_test")
    subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=undefined",
                    "-I", os.path.join(ROOT, "hunyuansc25_amd", "csrc"),
                    os.path.join(HERE, "native", "batch_plan_test.cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == "ok"
