"""Wave-per-query traversals at the edges of the wave tree's groups (64
leaves, 64 groups, 262 144 leaves per top group): neighbour lists against the
exact oracle, and against sorted FP64 distances where the oracle's full scan
would be long."""

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
