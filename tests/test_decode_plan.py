"""The decode kernels' work division (air.rs_amd/csrc/kernels/decode_plan.hpp) and
the key tiles of the f32-precision prefill (prefill_tiles.hpp), on the CPU: each
check in tests/*_check.cpp includes its header unchanged and builds with g++ here.
The first walks the pieces of random batches, the second compares sequences of up
to 2^31 - 1 keys with 64-bit arithmetic."""
import os
import shutil
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "air.rs_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("name", ["decode_plan_check", "prefill_tiles_check"])
def test_work_division(name):
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, name)
        subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-fsanitize=undefined", "-fno-sanitize-recover=undefined",
                        "-I", CSRC, "-o", exe, os.path.join(HERE, name + ".cpp")], check=True)
        out = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        print(out.stdout)
        assert out.returncode == 0, out.stdout + out.stderr
        assert ", 0 wrong" in out.stdout
