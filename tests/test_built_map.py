"""A context's kept tables (ciflow_amd/csrc/built_map.h) on the CPU: a table
whose construction fails part way is not kept.  Compiled with g++ under
AddressSanitizer + UndefinedBehaviorSanitizer."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = os.path.join(ROOT, "tests", "sanitize", "built_map_checks.cpp")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_half_made_tables_are_not_kept(tmp_path):
    exe = tmp_path / "built_map_checks"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-g", "-fsanitize=address,undefined", "-fno-sanitize-recover=all",
                        "-o", str(exe), SOURCE], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=1:verify_asan_link_order=0")
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300, env=env)
    assert r.returncode == 0 and "all kept table checks passed" in r.stdout, (r.stdout + r.stderr)[-6000:]


@pytest.mark.parametrize("source", ["capi.cpp", "solve_batch.cpp"])
def test_kept_tables_are_entered_through_it(source):
    """No subscript that makes an entry of a context's table map before its tables."""
    with open(os.path.join(ROOT, "ciflow_amd", "csrc", source)) as f:
        text = f.read()
    assert "doci_tabs[" not in text and "doci_blk[" not in text
