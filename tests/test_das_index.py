"""The delay-and-sum kernels' index and fixed-point arithmetic (ffdas_amd/csrc/das_index.h) run on the
CPU under UndefinedBehaviorSanitizer: scalar offsets inside a channel's block, every voxel in one
tile of every shape, the orders over the XCDs as bijections."""
import os
import shutil
import subprocess
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent / "asan"


def test_index_arithmetic():
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    r = subprocess.run(["make", "-C", str(HERE), "_build/index_asan"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0:halt_on_error=1:verify_asan_link_order=0",
               UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1")
    r = subprocess.run([str(HERE / "_build" / "index_asan")], capture_output=True, text=True, env=env,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "index arithmetic clean" in r.stdout
    assert "runtime error" not in r.stderr, r.stderr
