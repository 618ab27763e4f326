"""The order in which workgroups take pieces is a permutation that gives each XCD whole runs."""

import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_order_is_a_permutation_in_runs(tmp_path):
    cxx = shutil.which("g++")
    if not cxx:
        pytest.skip("g++ is needed to build the host check")
    exe = tmp_path / "xcd_order"
    r = subprocess.run([cxx, "-O2", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "elasticmegatron_amd", "csrc"),
                        os.path.join(ROOT, "tests", "native", "xcd_order.cpp"), "-o", str(exe)],
                       capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.returncode
    assert int(r.stdout.split()[1]) > 100_000
