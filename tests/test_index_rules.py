"""The kernels' index rules on the host (tests/cpp/index_check.cpp over
gadgetron_amd/csrc/gt_index.h): for every entry count of a chunk, a lane reads a
word of its own kind -- a sample index or a row mask -- inside the chunk's entries.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPP = os.path.join(ROOT, "tests", "cpp")


def test_index_rules():
    r = subprocess.run(["make", "-s", "-C", CPP, os.path.join(CPP, "index_check")], capture_output=True, text=True)
    if r.returncode == 127 or "not found" in r.stderr:
        pytest.skip("no host C++ compiler")
    assert r.returncode == 0, r.stderr
    r = subprocess.run([os.path.join(CPP, "index_check")], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout
