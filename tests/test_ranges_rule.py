"""Merged ranges of the direct backend and their mapped addresses, on the CPU
(tests/native/ranges_rule.cpp)."""

import os
import shutil
import subprocess

import pytest

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def test_a_range_is_mapped_only_where_all_of_it_is(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = tmp_path / "ranges_rule"
    proc = subprocess.run(["g++", "-std=c++20", "-O2", "-Wall", "-Wextra", "-Werror",
                           os.path.join(NATIVE, "ranges_rule.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout == "all ok\n", out.stdout
