"""Copies through the page-locked ring (csrc/pm_xfer.cpp) on the CPU, over a model of
the runtime calls it makes (tests/cpp/host_link): every line of its layout, pieces of
several segments, no page-locked or heap memory, and copy threads that sleep while an upload
waits for its stream."""
import os
import subprocess

import pytest

import __graft_entry__ as entry

HERE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "host_link")
CSRC = os.path.join(entry.PKG_DIR, "csrc")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("host_link") / "test_host_link")
    subprocess.check_call(["g++", "-O2", "-std=c++17", "-Wall", "-I", HERE, "-I", CSRC, "-o", out,
                           os.path.join(HERE, "test_host_link.cpp"),
                           os.path.join(CSRC, "pm_xfer.cpp"), "-pthread"])
    return out


@pytest.mark.parametrize("check", ["sizes", "lone", "parts", "no_ring", "no_heap", "sleeps"])
def test_host_link(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0, r.stdout + r.stderr
