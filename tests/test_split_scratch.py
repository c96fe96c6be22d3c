"""The buffers of split-k partitions, on the CPU against a model of HIP
(native/split_scratch_check.cpp): nothing that HIP refuses is called while a
stream is captured, a graph's buffer is its own and is never freed, the pool is
bounded, and without memory the product is told to make one pass."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from tests.conftest import ROOT


def test_partition_buffers_and_capture(tmp_path):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    exe = tmp_path / "check"
    subprocess.run([cxx, "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-DBLIS_IS_BUILDING_LIBRARY", "-I/opt/rocm/include", f"-I{ROOT / 'include'}",
                    str(ROOT / "tests" / "native" / "split_scratch_check.cpp"), "-o", str(exe),
                    "-lpthread"], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and p.stdout.strip() == "ok", p.stdout + p.stderr
