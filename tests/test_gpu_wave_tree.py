"""Wave-per-query traversals at the edges of the wave tree's groups (64
leaves, 64 groups, 262 144 leaves per top group): neighbour lists against the
exact oracle, and against sorted FP64 distances where the oracle's full scan
would be long."""

import time

import numpy as np
import pytest

import oracle
from helpers import mhgp, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k", [(2, 1), (5, 4), (33, 32), (63, 7), (64, 1), (65, 32), (129, 31), (4096, 5), (4097, 32)])
def test_neighbour_lists_at_group_edges(n, k):
    pts = workloads.uniform_cloud(n, seed=n)
    canon = oracle.canonicalize(pts)
    print(f"wave tree: knn n={n} k={k}", flush=True)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        ids = ctx.knn(k)
    ref, _ = oracle.knn(canon, k)
    assert np.array_equal(ids.astype(np.int64), ref)


@pytest.mark.parametrize("offset", [0.0, 1.0e6])
def test_neighbour_lists_across_top_groups(offset):
    n, k = 262_144 + 70, 9
    pts = workloads.uniform_cloud(n, seed=3) + offset
    print(f"wave tree: knn n={n} offset {offset}", flush=True)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        xyz, _ = ctx.canonical_points()
        ids = ctx.knn(k)
    for u in np.random.default_rng(0).integers(0, n, size=64):
        d = ((xyz - xyz[u]) ** 2).sum(1)
        d[u] = np.inf
        near = np.argsort(d, kind="stable")[: k + 1]
        # distances of a random cloud are distinct far beyond the rounding of the sums
        assert np.array_equal(ids[u], near[:k]), u


def test_a_far_outlier_does_not_slow_the_others():
    """One point a million times the cloud's extent away: the boxes still tell
    the others apart.  (Where they cannot, each query looks at every point: 25
    times as long at this size.  The outlier itself costs about a factor of two:
    the others share a few Morton cells, so their groups are slabs.)"""
    n, k = 200_000, 8
    pts = workloads.uniform_cloud(n, seed=12)
    far = pts.copy()
    far[5] = [1.0e6, 0.0, 0.0]
    print(f"wave tree: knn n={n} with a far outlier", flush=True)
    best = []
    for cloud in (pts, far):
        with mhgp.Context(0) as ctx:
            ctx.upload(cloud)
            times = []
            for _ in range(5):
                start = time.perf_counter()
                ids = ctx.knn(k)
                times.append(time.perf_counter() - start)
            xyz, _ = ctx.canonical_points()
        best.append(min(times))
    print(f"without {best[0] * 1e3:.2f} ms, with {best[1] * 1e3:.2f} ms", flush=True)
    for u in np.random.default_rng(1).integers(0, n - 1, size=8):
        d = ((xyz - xyz[u]) ** 2).sum(1)
        d[u] = np.inf
        assert np.array_equal(ids[u], np.argsort(d, kind="stable")[:k]), u
    assert best[1] < 6.0 * best[0]
