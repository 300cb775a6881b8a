"""The FP64 level of a record is a function of its support alone: every record
of a catalogue, from whichever kernel it came, has the bits that the same
expressions (e-hgp_amd/csrc/predicates.hpp) give on the host."""

import ctypes
import os
import subprocess

import numpy as np
import pytest

from helpers import PKG, mhgp, workloads

HERE = os.path.dirname(os.path.abspath(__file__))

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def host_levels(tmp_path_factory):
    out = tmp_path_factory.mktemp("levels") / "liblevels.so"
    cmd = ["/opt/rocm/bin/hipcc", "-O2", "-ffp-contract=off", "-fPIC", "-shared", "-std=c++17", "-D__HIP_PLATFORM_AMD__",
           "-x", "c++", "-I", os.path.join(PKG, "csrc"), "-I/opt/rocm/include",
           os.path.join(HERE, "native", "level_check.cpp"), "-o", str(out)]
    subprocess.run(cmd, check=True, capture_output=True)
    lib = ctypes.CDLL(str(out))
    p = ctypes.c_void_p
    lib.levels.argtypes = [p, p, ctypes.c_long, p]

    def run(xyz, ids, size):
        rel = np.zeros((len(ids), 9))
        for j in (1, 2, 3):
            has = size > j
            rel[has, 3 * (j - 1): 3 * j] = xyz[ids[has, j]] - xyz[ids[has, 0]]
        size = np.ascontiguousarray(size, dtype=np.int32)
        got = np.zeros(len(ids))
        lib.levels(rel.ctypes.data, size.ctypes.data, len(ids), got.ctypes.data)
        return got

    return run


@pytest.mark.parametrize("name", ["lattice", "mixture", "nearly_regular", "slabs"])
def test_level_is_a_function_of_the_support(name, host_levels, monkeypatch):
    k = 10
    if name == "lattice":
        pts = workloads.jittered_lattice(1000, side=11, sigma=0.1, seed=5)
    elif name == "nearly_regular":
        pts, k = workloads.jittered_lattice(500, side=8, sigma=1e-2, seed=5), 8
    else:
        pts = workloads.gaussian_mixture(1000, blobs=5, noise_fraction=0.15, box=10.0, snap_bits=None, seed=4)
        if name == "slabs":
            monkeypatch.setenv("MHGP_TEST_ANCHOR_PATH", "slabs")
            pts, k = pts[:300], 6
    print(f"levels: {name} n={len(pts)} k={k}", flush=True)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        got = ctx.supports_raw(k)
        xyz, _ = ctx.canonical_points()
    assert got["info"].fallback_count == 0  # the host's records have the exact ratio instead
    want = host_levels(xyz, got["ids"].astype(np.int64), got["meta"] & 0xFF)
    assert np.array_equal(got["level"], want), int((got["level"] != want).sum())
