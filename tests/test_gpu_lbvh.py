"""Canonical cloud, exact Morton LBVH snapshot and k-NN on the GPU vs the oracle."""

import time

import numpy as np
import pytest

import oracle
from helpers import mhgp, workloads

pytestmark = pytest.mark.gpu


def _clouds():
    rng = np.random.default_rng(123)
    yield "single", np.array([[0.5, -0.0, 2.0]])
    yield "pair", np.array([[1.0, 2.0, 3.0], [-1.0, 2.0, 3.0]])
    yield "uniform17", rng.random((17, 3))
    yield "uniform1000", workloads.uniform_cloud(1000, seed=3)
    yield "lattice3000", workloads.jittered_lattice(3000, side=16, seed=4)
    grid = np.stack(np.meshgrid(np.arange(6), np.arange(6), np.arange(6)), -1).reshape(-1, 3) * 0.25
    yield "exact_grid216", grid.astype(float)
    # runs of equal Morton codes (bin width 2^-21 of the extent): midpoint splits
    run = [[i * 1e-9, (i % 3) * 1e-9, 0.0] for i in range(7)]
    run += [[0.5 + i * 1e-9, 0.5, 0.5] for i in range(6)]
    tiny = np.array(run + [[1.0, 1.0, 1.0], [0.25, 0.75, 0.1]], dtype=float)
    yield "equal_codes", tiny
    yield "mixture2000", workloads.gaussian_mixture(2000, blobs=5, seed=5)


@pytest.mark.parametrize("name,pts", list(_clouds()), ids=lambda v: v if isinstance(v, str) else "")
def test_canonical_and_snapshot_match_oracle(name, pts):
    print(f"case {name} n={len(pts)}", flush=True)
    canon = oracle.canonicalize(pts)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        xyz, src = ctx.canonical_points()
        assert np.array_equal(xyz, canon)
        assert np.array_equal(np.asarray(pts)[src] + 0.0, canon)
        leaves, nodes, counters = ctx.lbvh_snapshot()
        ref = oracle.lbvh_snapshot(canon)
        assert np.array_equal(leaves, ref.leaves)
        assert np.array_equal(nodes, ref.nodes)
        assert np.array_equal(counters, ref.counters)


def test_knn_matches_oracle():
    for name, pts in _clouds():
        if len(pts) < 12 or len(pts) > 3000:
            continue
        print(f"knn case {name}", flush=True)
        canon = oracle.canonicalize(pts)
        with mhgp.Context(0) as ctx:
            ctx.upload(pts)
            for k in (1, 11, 32):
                if k >= len(pts):
                    continue
                ids = ctx.knn(k)
                ref, _ = oracle.knn(canon, k)
                assert np.array_equal(ids.astype(np.int64), ref), (name, k)


def test_rejects_duplicates_and_nonfinite():
    with mhgp.Context(0) as ctx:
        with pytest.raises(mhgp.MhgpError) as e:
            ctx.upload([[0, 0, 0], [1, 1, 1], [0, -0.0, 0]])
        assert e.value.code == mhgp.E_DUPLICATE
        with pytest.raises(mhgp.MhgpError) as e:
            ctx.upload([[0, 0, 0], [np.nan, 1, 1]])
        assert e.value.code == mhgp.E_NONFINITE
        ctx.upload([[0, 0, 0], [1, 1, 1]])  # context stays usable after argument errors
        assert ctx.n == 2


def test_lattice_50k_snapshot_invariants():
    pts = workloads.jittered_lattice(50_000, seed=0)
    canon = oracle.canonicalize(pts)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        leaves, nodes, counters = ctx.lbvh_snapshot()
    ref = oracle.lbvh_snapshot(canon)
    assert np.array_equal(leaves, ref.leaves)
    assert np.array_equal(nodes, ref.nodes)
    # published snapshot size of the reference at n = 50 000: 176 n - 80 bytes
    assert leaves.nbytes + nodes.nbytes == 176 * 50_000 - 80


def test_device_snapshot_is_certified_exactly():
    """The device snapshot passes the exact host re-certification (the
    reference's import_certified_snapshot role) at 50 000 points and on a
    cloud with equal-code runs."""
    for label, pts in (("lattice50k", workloads.jittered_lattice(50_000, side=37, seed=0)),
                       ("collisions", np.concatenate([workloads.uniform_cloud(200, seed=3),
                                                      0.5 + np.arange(40)[:, None] * 1e-13 * np.ones((1, 3))]))):
        print(f"certify device snapshot {label}", flush=True)
        with mhgp.Context(0) as ctx:
            ctx.upload(pts)
            xyz, _ = ctx.canonical_points()
            leaves, nodes, counters = ctx.lbvh_snapshot()
        mhgp.lbvh_certify(xyz, leaves, nodes, counters)


def _build_edges():
    """Sizes around the one-workgroup sort and the sort tiles, and clouds whose
    coarse canonical keys collide: tight clusters (short runs, repaired), a far
    outlier that puts every other point into one run and columns of equal x
    (the sort of the full coordinates), and signed zeros."""
    for n in (2, 63, 65, 4096, 4097, 8192, 8193):
        yield f"uniform{n}", workloads.uniform_cloud(n, seed=n)
    rng = np.random.default_rng(8)
    centres = rng.random((700, 3))
    yield "clusters", np.repeat(centres, 13, axis=0) + rng.normal(0.0, 1e-9, size=(9100, 3))
    far = workloads.uniform_cloud(9000, seed=4)
    far[17] = [1e12, -1e12, 1e12]
    yield "outlier", far
    cols = rng.random((9000, 3))
    cols[:, 0] = np.floor(cols[:, 0] * 4) / 4 + rng.random(9000) * 1e-12
    yield "columns", cols
    zero = workloads.uniform_cloud(300, seed=5) - 0.5
    zero[:40, 0] = np.where(np.arange(40) % 2, 0.0, -0.0)
    yield "zeros", zero


@pytest.mark.parametrize("name,pts", list(_build_edges()), ids=lambda v: v if isinstance(v, str) else "")
def test_build_at_its_edges(name, pts):
    print(f"build edge case {name} n={len(pts)}", flush=True)
    canon = oracle.canonicalize(pts)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        xyz, src = ctx.canonical_points()
        assert np.array_equal(xyz, canon)
        assert np.array_equal(np.asarray(pts)[src] + 0.0, canon)
        leaves, nodes, counters = ctx.lbvh_snapshot()
    ref = oracle.lbvh_snapshot(canon)
    assert np.array_equal(leaves, ref.leaves)
    assert np.array_equal(nodes, ref.nodes)
    assert np.array_equal(counters, ref.counters)


@pytest.mark.parametrize("runs", [[], [2], [3, 2], [5, 700, 2, 64], [4097]])
def test_snapshot_totals_of_equal_codes(runs):
    """The snapshot's collision totals (runs of equal codes, the longest) and
    canonical points against the fetched arrays: runs of many lengths, each a
    cluster within one Morton cell, beside points that share no cell."""
    rng = workloads.SplitMix64(77 + len(runs)).numpy_rng()
    parts = [rng.uniform(0.0, 1.0, size=(300, 3))]
    for r in runs:
        parts.append(rng.uniform(0.1, 0.9, size=(1, 3)) + rng.uniform(0.0, 1e-12, size=(r, 3)))
    pts = np.concatenate(parts)
    print(f"snapshot totals: runs {runs}", flush=True)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        leaves, nodes, counters = ctx.lbvh_snapshot()
        xyz, source = ctx.canonical_points()
    _, lengths = np.unique(leaves[:, 0], return_counts=True)
    long = lengths[lengths > 1]
    assert list(counters[:2]) == [len(xyz), 2 * len(xyz) - 1]
    assert counters[3] == len(long) and counters[4] == (long.max() if len(long) else 0)
    assert np.array_equal(xyz, pts[source])
    # depth from the postorder nodes' children
    depth = np.zeros(len(nodes), dtype=np.int64)
    for i in range(len(nodes) - 1, -1, -1):
        for child in nodes[i, 6:8]:
            if child != 0xFFFFFFFFFFFFFFFF:
                depth[int(child)] = depth[i] + 1
    assert counters[2] == depth.max()


def test_a_run_that_needs_the_full_sort_is_not_built_twice():
    """Half the points in one cell of the coarse key: in lexicographic source
    order the coarse sort leaves them in order, shuffled they need the sort of
    the full coordinates.  That sort costs a few tenths of a millisecond; the
    leaves of equal codes (milliseconds here) must not be made for both."""
    rng = np.random.default_rng(4)
    pts = rng.uniform(size=(50_000, 3))
    pts[:25_000] *= 1e-8
    pts = pts[np.lexsort((pts[:, 2], pts[:, 1], pts[:, 0]))]
    print("upload of 25 000 points in one cell, in order and shuffled", flush=True)
    best = []
    for cloud in (pts, pts[rng.permutation(len(pts))]):
        with mhgp.Context(0) as ctx:
            times = []
            for _ in range(8):
                start = time.perf_counter()
                ctx.upload(cloud)
                times.append(time.perf_counter() - start)
            xyz, _ = ctx.canonical_points()
        assert np.array_equal(xyz, pts)
        best.append(min(times))
    print(f"in order {best[0] * 1e3:.2f} ms, shuffled {best[1] * 1e3:.2f} ms", flush=True)
    assert best[1] < 1.4 * best[0]
