"""The cache of temporaries: eviction, limits per device, memory that runs
out, threads (tests/cpp/test_tmp_cache.cpp, over a counting allocator)."""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host C++ compiler")
def test_tmp_cache(tmp_path):
    exe = tmp_path / "test_tmp_cache"
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-pthread",
                        f"-I{ROOT / 'morpheus_amd' / 'csrc'}", "-o", str(exe),
                        str(ROOT / "tests" / "cpp" / "test_tmp_cache.cpp")],
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout[-4000:]
