"""The cache of temporaries: eviction, limits per device, memory that runs
out, threads (tests/cpp/test_tmp_cache.cpp, over a counting allocator)."""
import re
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


def test_allocations_may_ask_for_the_temporaries():
    """Plans, batches, solvers and containers allocate through the functions
    that give the held temporaries back when memory has run out."""
    csrc = ROOT / "morpheus_amd" / "csrc"
    for f in sorted(csrc.glob("*.hip")) + sorted(csrc.glob("*.hpp")) + sorted(csrc.glob("*.cpp")):
        text = re.sub(r"//.*", "", f.read_text())
        assert len(re.findall(r"\bhipMalloc\w*\(", text)) == (2 if f.name == "capi.cpp" else 0), f
    for f in sorted((ROOT / "morpheus_amd" / "include").glob("*.hpp")):
        # (the two tries of device_malloc)
        text = re.sub(r"//.*", "", f.read_text())
        assert text.count("hipMalloc(") == (2 if "device_malloc(void** p" in text else 0), f


def test_container_allocation_asks_for_the_temporaries(monkeypatch):
    import torch

    from morpheus_amd import capi, device
    asked, tries, empty = [], [], torch.empty

    def full(*a, device=None, **k):
        tries.append(a)
        if len(tries) == 1:
            raise torch.OutOfMemoryError("full")
        return empty(*a, **k)

    monkeypatch.setattr(torch, "empty", full)
    monkeypatch.setattr(capi, "call", lambda name, *a: asked.append(name))
    assert device._empty_i(7).numel() == 7 and asked == ["mph_finalize"] and len(tries) == 2
