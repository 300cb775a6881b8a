"""The server admits a request by its predicted device memory
(e-hgp_amd/csrc/budget.hpp): the prediction covers what the catalogue
allocates before it has seen a record, and what a context holds after a
whole request."""

import ctypes
import os
import subprocess

import pytest

from helpers import PKG, mhgp, workloads

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    out = tmp_path_factory.mktemp("budget") / "libbudget.so"
    subprocess.run(["g++", "-O1", "-fPIC", "-shared", "-std=c++17", "-Wall", "-Werror", "-I", os.path.join(PKG, "csrc"),
                    os.path.join(HERE, "native", "budget_check.cpp"), "-o", str(out)], check=True, capture_output=True)
    lib = ctypes.CDLL(str(out))
    for f in (lib.budget_predict, lib.budget_catalogue, lib.budget_queues, lib.budget_bounded):
        f.argtypes = [ctypes.c_int64, ctypes.c_int]
        f.restype = ctypes.c_int64
    lib.budget_slabs.argtypes = [ctypes.c_int64, ctypes.c_uint64, ctypes.c_int64, ctypes.c_int64]
    lib.budget_slabs.restype = ctypes.c_uint64
    return lib


@pytest.mark.parametrize("n", [1, 64, 1000, 17117, 50000, 200000, 2000000])
def test_prediction_covers_the_first_allocations(lib, n):
    for k in range(1, 11):
        rows = n * (64 * 4 + 9)  # a tower's neighbour rows
        assert lib.budget_predict(n, k) >= lib.budget_catalogue(n, k) + rows
        assert lib.budget_predict(n, k) >= lib.budget_predict(n, max(k - 1, 1))


@pytest.mark.parametrize("n", [2, 7, 64, 1000, 16384, 16385, 17117, 50000, 2000000])
def test_bounded_queues_leave_room_for_slabs_and_rescans(lib, n):
    """With rescans, the slabs' least, the tables (53 248 bytes) and the wider
    rows and lists (138 bytes a point) the queues of a context with a device
    capacity take no more than the plain queues."""
    for k in range(1, 11):
        assert lib.budget_bounded(n, k) + 53248 + 138 * n <= lib.budget_queues(n, k)


def test_slabs_grow_into_a_quarter_of_what_is_left(lib):
    mib = 1 << 20
    assert lib.budget_slabs(400 * mib, 0, mib, 2048 * mib) == 100 * mib
    assert lib.budget_slabs(400 * mib, 50 * mib, mib, 2048 * mib) == 150 * mib
    assert lib.budget_slabs(0, 0, mib, 2048 * mib) == mib
    assert lib.budget_slabs(-5, 0, mib, 2048 * mib) == mib
    assert lib.budget_slabs(1 << 40, 0, mib, 2048 * mib) == 2048 * mib
    assert lib.budget_slabs(0, 0, 4096 * mib, 2048 * mib) == 2048 * mib


@pytest.mark.gpu
@pytest.mark.parametrize("n,k,tower", [(256, 3, True), (1000, 10, True), (5000, 4, True), (17117, 4, False)])
def test_a_request_holds_what_was_predicted(lib, n, k, tower):
    """Measured: a jittered lattice through a fresh context (a server's slot
    has one tower lane, this context more of them)."""
    side = int((n * 1.01) ** (1 / 3)) + 1
    print(f"prediction: lattice n={n} k={k}", flush=True)
    with mhgp.Context(0) as ctx:
        ctx.upload(workloads.jittered_lattice(n, side=side, sigma=0.1, seed=2))
        ctx.emst()
        info = ctx.supports(k, fetch=False)
        assert info.status == 0
        if tower:
            ctx.tower(k, fetch=False)
        held = ctx.device_bytes()
    assert held <= lib.budget_predict(n, k), (held, lib.budget_predict(n, k))
