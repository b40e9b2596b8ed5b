"""Fragments cut into 16-byte chunks: the rule and the arithmetic that the copy
kernels share with the host, on the CPU (tests/native/chunk_rule.cpp)."""

import os
import shutil
import subprocess

import pytest

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")


def test_chunks_cover_every_fragment_they_are_used_for(tmp_path):
    """Sizes around 2 GiB, 4 GiB and beyond among them: a fragment whose length
    does not fit the chunk arithmetic keeps to tiles."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = tmp_path / "chunk_rule"
    proc = subprocess.run(["g++", "-std=c++20", "-O2", "-Wall", "-Wextra", "-Werror",
                           os.path.join(NATIVE, "chunk_rule.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout == "all ok\n", out.stdout


def test_chunks_along_the_links_packets_cover_a_range(tmp_path):
    """tests/native/lines_rule.cpp: fragments from 16 bytes on, every start modulo 256."""
    if shutil.which("g++") is None:
        pytest.skip("g++ not installed")
    exe = tmp_path / "lines_rule"
    proc = subprocess.run(["g++", "-std=c++20", "-O2", "-Wall", "-Wextra", "-Werror",
                           os.path.join(NATIVE, "lines_rule.cpp"), "-o", str(exe)], capture_output=True, text=True)
    assert proc.returncode == 0, proc.stderr
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0 and out.stdout == "all ok\n", out.stdout
