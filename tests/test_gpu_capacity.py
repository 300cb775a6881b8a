"""Contexts with a device capacity: the slabs, anchor lists and rescans of the
enumeration are fitted into what the record queues and the tower's workspaces
leave, so that a capacity which held those alone (the bytes below, measured
with an enumeration that had no slabs) takes the same clouds."""

import numpy as np
import pytest

from helpers import mhgp, workloads

pytestmark = pytest.mark.gpu


def _cloud(kind, n):
    if kind == "lattice":
        return workloads.jittered_lattice(n, side=int((n * 1.01) ** (1 / 3)) + 1, sigma=0.1, seed=1)
    if kind == "uniform":
        return workloads.uniform_cloud(n, seed=1)
    return workloads.gaussian_mixture(n, blobs=5, noise_fraction=0.15, box=10.0, snap_bits=None, seed=1)


CASES = [("uniform", 64, 3, 5596676, 5868848), ("uniform", 256, 3, 9424320, 10693096),
         ("lattice", 1000, 1, 15167636, 16111196), ("lattice", 1000, 4, 28991636, 41679256),
         ("mixture", 1000, 10, 54789264, 89469028), ("lattice", 5000, 4, 128558552, 202129136),
         ("mixture", 2003, 4, 178247362, 197058566), ("lattice", 17117, 4, 432081074, 706983882)]


@pytest.mark.parametrize("kind,n,k,catalogue,tower", CASES)
def test_capacity_of_queues_and_workspaces_is_enough(kind, n, k, catalogue, tower):
    pts = _cloud(kind, n)
    print(f"capacity: {kind} n={n} k={k}", flush=True)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        ref = ctx.supports_raw(k)
        ref_tower = ctx.tower(k)
    with mhgp.Context(0, capacity_bytes=catalogue) as ctx:
        ctx.upload(pts)
        ctx.emst()
        got = ctx.supports_raw(k)
        assert ctx.device_bytes() <= catalogue
    for key in ("ids", "meta", "interior", "level", "level_class"):
        assert np.array_equal(got[key], ref[key]), key
    with mhgp.Context(0, capacity_bytes=catalogue) as ctx:
        ctx.upload(pts)
        ctx.supports(k, fetch=False)
        ctx.emst()  # its buffers after the catalogue's
        assert ctx.device_bytes() <= catalogue
    with mhgp.Context(0, capacity_bytes=tower) as ctx:
        for _ in range(2):  # the second time beside the workspaces of the first
            ctx.upload(pts)
            ctx.emst()
            ctx.supports(k, fetch=False)
            got_tower = ctx.tower(k)
            got = ctx.supports_raw(k) if _ else ref
            assert ctx.device_bytes() <= tower
            for key in ("order", "kind", "level_class", "level", "child_offset", "children", "vertical"):
                assert np.array_equal(got_tower[key], ref_tower[key]), key
    for key in ("ids", "meta", "interior", "level", "level_class"):
        assert np.array_equal(got[key], ref[key]), key


def test_rescans_of_a_nearly_regular_cloud_fit_at_once(capfd, monkeypatch):
    """Lattices displaced by 1% of their spacing leave several sides a point to
    the rescans: where the capacity has room for them the list does not start
    at one a point, which would run the enumeration twice."""
    n = 6000
    pts = workloads.jittered_lattice(n, side=19, sigma=0.01, seed=5)
    monkeypatch.setenv("MHGP_TIMING", "1")
    print(f"capacity: nearly regular lattice n={n}", flush=True)
    with mhgp.Context(0, capacity_bytes=4 << 30) as ctx:
        ctx.upload(pts)
        capfd.readouterr()
        ctx.supports(10, fetch=False)
    lines = [ln for ln in capfd.readouterr().err.splitlines() if "sides left to the rescans" in ln]
    most = int(lines[-1].split()[-1])
    assert most > max(1 << 14, n), "the cloud no longer leaves sides to the rescans"
    assert len(lines) == 1  # one run of the enumeration
