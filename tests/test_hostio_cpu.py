"""Pinned-slot transfers (opendxmc_amd/csrc/hostio.cpp) on a stand-in for the
HIP runtime: pinned memory or threads refused, other current devices.
tests/cpp/hostio_check.cpp, one case a test."""
from __future__ import annotations

import subprocess
from pathlib import Path

import pytest

from opendxmc_amd import build


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = tmp_path_factory.mktemp("hostio") / "hostio_check"
    rocm = Path(build.HIPCC).resolve().parent.parent
    subprocess.run(["g++", "-std=c++17", "-O2", "-D__HIP_PLATFORM_AMD__", f"-I{build.CSRC}", "-isystem", str(rocm / "include"),
                    str(build.TESTS_CPP / "hostio_check.cpp"), str(build.CSRC / "hostio.cpp"), "-pthread", "-ldl", "-o", str(exe)],
                   check=True, timeout=120)
    return exe


@pytest.mark.parametrize("case", ["plain", "pinned memory refused", "threads refused", "stream of another device", "earlier error", "waiting"])
def test_transfers(program, case):
    r = subprocess.run([str(program), case], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
