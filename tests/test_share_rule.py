"""The share of a staging fill that crosses the link with its gather or scatter
launch: where the fill is cut, on the CPU (tests/native/share_rule.cpp)."""

import os
import shutil
import subprocess

import pytest

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def test_cut_of_a_fill_leaves_its_tail(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = tmp_path / "share_rule"
    proc = subprocess.run(["g++", "-std=c++20", "-O2", "-Wall", "-Wextra", "-Werror",
                           os.path.join(NATIVE, "share_rule.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout == "all ok\n", out.stdout
