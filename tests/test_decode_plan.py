"""The decode kernels' work division (air.rs_amd/csrc/kernels/decode_plan.hpp),
on the CPU: tests/decode_plan_check.cpp includes that header unchanged, builds
with g++ here and walks the pieces of random batches."""
import os
import shutil
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "air.rs_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_decode_plan():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "decode_plan_check")
        subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", CSRC, "-o", exe,
                        os.path.join(HERE, "decode_plan_check.cpp")], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        print(out.stdout)
        assert out.returncode == 0, out.stdout
        assert ", 0 wrong" in out.stdout
