"""The device-block cache's policy (ciflow_amd/csrc/block_cache.h) on the CPU,
compiled with g++ under AddressSanitizer + UndefinedBehaviorSanitizer and under
ThreadSanitizer."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "tests", "sanitize", "block_cache_checks.cpp")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("sanitizer", ["address,undefined", "thread"])
def test_block_cache_policy(tmp_path, sanitizer):
    exe = tmp_path / "block_cache_checks"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-pthread", f"-fsanitize={sanitizer}",
                        "-fno-sanitize-recover=all", "-o", str(exe), SOURCE], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:verify_asan_link_order=0")
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300, env=env)
    assert r.returncode == 0 and "all block cache checks passed" in r.stdout, (r.stdout + r.stderr)[-6000:]
