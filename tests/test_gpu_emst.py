"""Exact Borůvka EMST on the GPU vs the oracle's complete-graph Kruskal."""

from fractions import Fraction

import numpy as np
import pytest

import oracle
from helpers import mhgp, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("name", ["uniform500", "lattice2000", "grid_ties", "mixture1500", "square_tail"])
def test_emst_matches_kruskal(name):
    print(f"emst case {name}", flush=True)
    if name == "uniform500":
        pts = workloads.uniform_cloud(500, seed=11)
    elif name == "lattice2000":
        pts = workloads.jittered_lattice(2000, side=13, seed=12)
    elif name == "grid_ties":  # exact equal squared lengths everywhere
        g = np.stack(np.meshgrid(np.arange(7), np.arange(7), np.arange(7)), -1).reshape(-1, 3)
        pts = g.astype(float) * 0.5
    elif name == "mixture1500":
        pts = workloads.gaussian_mixture(1500, blobs=4, seed=13)
    else:
        pts = np.array([[-1, -1, 0], [-1, 1, 0], [1, -1, 0], [1, 1, 0], [5, 0, 0]], dtype=float)
    canon = oracle.canonicalize(pts)
    ref = oracle.emst(canon)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        e = ctx.emst().astype(np.int64)
    assert np.array_equal(e, ref)


@pytest.mark.parametrize("name", ["two", "group64", "group65", "level4097", "chain", "near_ties", "far_away"])
def test_emst_rounds_at_their_edges(name):
    """Group and level edges of the wave tree, a chain whose components all
    hook one way (the longest hook path), tied lengths that FP64 cannot prove
    (settled on the host), and a cloud far from the origin."""
    print(f"emst edge case {name}", flush=True)
    if name in ("two", "group64", "group65", "level4097"):
        n = {"two": 2, "group64": 64, "group65": 65, "level4097": 4097}[name]
        pts = workloads.uniform_cloud(n, seed=n)
    elif name == "chain":
        step = 1.0 + 1e-3 * np.arange(2500)
        pts = np.stack([np.cumsum(step), np.zeros(2500), np.zeros(2500)], axis=1)
    elif name == "near_ties":
        pts = np.stack(np.meshgrid(np.arange(6), np.arange(6), np.arange(6)), -1).reshape(-1, 3) * 0.1
    else:
        pts = workloads.uniform_cloud(1500, seed=4) + 1.0e7
    ref = oracle.emst(oracle.canonicalize(pts))
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        e = ctx.emst().astype(np.int64)
    assert np.array_equal(e, np.asarray(ref, dtype=np.int64).reshape(e.shape))


def _sq(q):  # squared length, rounded as the device does
    return (q[0] * q[0] + q[1] * q[1]) + q[2] * q[2]


def _kept_result_cloud():
    """Two points x, y whose FP64 distances to p (the origin) are one ulp
    apart in the order opposite to the exact one, and a point a of p's
    component whose own result, kept from the round before, lies just far
    enough below both that the first is within its rounding window and the
    second is not.  Clusters with doubling gaps let p, a and the others merge
    at smaller distances round by round until then."""
    x, y, w = [-0.8190404901453785, 6.425679486307635e-05, 0.5737357156160684], [-0.820664404928251, -0.0007032900117319003, -0.5714100452975243], 0.9999999999994997
    assert _sq(y) == np.nextafter(_sq(x), 2.0) and sum(Fraction(c) ** 2 for c in y) < sum(Fraction(c) ** 2 for c in x)
    assert w * w * (1.0 + 1e-12) + 1e-300 == _sq(x) and _sq(x) - w * w > 1e-12 * (w * w)
    pts = [[0, 0, 0], [0, 0.1, 0], [0, 0.45, 0], [0, 0.55, 0]]
    pts += [[0, -0.9 - o, 0] for o in (0, 0.1, 0.4, 0.5)]
    pts += [[w + o, 0.55, 0] for o in (0, 0.1, 0.4, 0.5, 1.1, 1.2, 1.5, 1.6)]
    turns = np.array([x, [-1.62, 0, x[2]], [-1.62, 0, y[2]], y])
    leg = np.linalg.norm(np.diff(turns, axis=0), axis=1)
    ends = np.concatenate([[0.0], np.cumsum(leg)])
    gaps = np.array([0.1, 0.2, 0.1, 0.3, 0.1, 0.2, 0.1, 0.4, 0.1, 0.2, 0.1, 0.3, 0.1, 0.2, 0.1])
    for s in np.cumsum(gaps)[:-1] * ends[-1] / gaps.sum():
        k = min(int(np.searchsorted(ends, s, side="right")) - 1, 2)
        pts.append(list(turns[k] + (turns[k + 1] - turns[k]) * (s - ends[k]) / leg[k]))
    return np.array(pts + [x, y], dtype=float)


def test_emst_near_ties_of_kept_results():
    """A search ends at the rounding window of its component's best offer; a
    near tie just beyond it still has to be known when the result is used in a
    later round, where that offer is gone."""
    pts = _kept_result_cloud()
    print("emst: near tie beyond an offer's window", flush=True)
    ref = oracle.emst(oracle.canonicalize(pts))
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        e = ctx.emst().astype(np.int64)
    assert np.array_equal(e, ref)


def test_emst_ties_of_absorbed_points_are_not_settled_again(capfd, monkeypatch):
    """The same cloud: only the two components of the last round hold a tie.
    Others' results tied in an earlier round with a point that has been
    absorbed since; the host (quadratic in the component) need not see them."""
    monkeypatch.setenv("MHGP_TIMING", "1")
    print("emst: ties of absorbed points", flush=True)
    with mhgp.Context(0) as ctx:
        ctx.upload(_kept_result_cloud())
        capfd.readouterr()
        ctx.emst()
    lines = [ln for ln in capfd.readouterr().err.splitlines() if "settled on the host" in ln]
    assert [int(ln.split()[-1]) for ln in lines] == [2]


def test_emst_50k_lattice_weight():
    from scipy.sparse import coo_matrix
    from scipy.sparse.csgraph import minimum_spanning_tree

    pts = workloads.jittered_lattice(50_000, seed=0)
    with mhgp.Context(0) as ctx:
        ctx.upload(pts)
        xyz, _ = ctx.canonical_points()
        e = ctx.emst().astype(np.int64)
        nb = ctx.knn(32).astype(np.int64)
    n = len(xyz)
    assert len(e) == n - 1 and np.all(e[:, 0] < e[:, 1])
    w = np.sqrt(((xyz[e[:, 0]] - xyz[e[:, 1]]) ** 2).sum(1))
    assert np.all(np.diff(w ** 2) >= -1e-12)  # kappa order
    rows = np.repeat(np.arange(n), 32)
    d = np.sqrt(((xyz[rows] - xyz[nb.ravel()]) ** 2).sum(1))
    g = coo_matrix((d, (rows, nb.ravel())), shape=(n, n)).tocsr()
    mst = minimum_spanning_tree(g)
    assert abs(mst.sum() - w.sum()) <= 1e-9 * w.sum()
    # spanning: union-find over the edges
    parent = np.arange(n)

    def find(x):
        while parent[x] != x:
            parent[x] = parent[parent[x]]
            x = parent[x]
        return x

    for a, b in e:
        ra, rb = find(a), find(b)
        assert ra != rb
        parent[ra] = rb
