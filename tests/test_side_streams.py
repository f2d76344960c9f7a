"""The pool of side streams (csrc/side.hip) on the CPU: compiled with g++ against stubs of the
HIP calls it makes. Callers on different streams get different side streams (one shared by
all made independent callers queue behind each other), a call never waits for another
thread, the pool is bounded, and a captured call runs unsplit."""

import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_side_streams(tmp_path):
    exe = str(tmp_path / "side_test")
    src = os.path.join(HERE, "native", "side_test.cpp")
    subprocess.run(["g++", "-std=c++17", "-O1", "-pthread", "-I", os.path.join(HERE, "native"), src, "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
