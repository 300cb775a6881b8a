"""Copies of a large tower run one thread an order.  Where the system refuses a
thread the order is copied by the caller; the process must not end
(tests/native/threads_check.cpp, whose pthread_create refuses)."""

import os
import subprocess

import pytest

from helpers import PKG

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("threads") / "threads_check"
    cmd = ["/opt/rocm/bin/hipcc", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-x", "c++", "-I", os.path.join(PKG, "csrc"),
           "-I/opt/rocm/include", os.path.join(HERE, "native", "threads_check.cpp"), "-o", str(out), "-pthread", "-ldl"]
    subprocess.run(cmd, check=True, capture_output=True)
    return str(out)


@pytest.mark.parametrize("allowed", [0, 1, 3, 100])
def test_copies_without_enough_threads(exe, allowed):
    r = subprocess.run([exe, str(allowed)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.strip() == "ok", (r.returncode, r.stdout, r.stderr)
