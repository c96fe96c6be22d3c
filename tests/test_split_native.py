"""Host code of split-k products, compiled and run on the CPU: the rule for the
partitions (native/split_rule_check.cpp), and their buffers against a model of HIP
(native/split_scratch_check.cpp): nothing that HIP refuses is called while a
stream is captured, a graph's buffer is its own and is never freed, the pool is
bounded, and without memory the product is told to make one pass."""
from __future__ import annotations

import shutil
import subprocess

import pytest

from tests.conftest import ROOT


@pytest.mark.parametrize("check", ["split_scratch_check", "split_rule_check"])
def test_native(tmp_path, check):
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    exe = tmp_path / "check"
    subprocess.run([cxx, "-std=c++17", "-O1", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-DBLIS_IS_BUILDING_LIBRARY", "-I/opt/rocm/include", f"-I{ROOT / 'include'}",
                    str(ROOT / "tests" / "native" / f"{check}.cpp"), "-o", str(exe),
                    "-lpthread"], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert p.returncode == 0 and p.stdout.strip() == "ok", p.stdout + p.stderr
