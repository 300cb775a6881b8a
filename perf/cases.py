"""Performance cases: the work a user of the library has it do, through the
Python binding's public entry points (e-hgp_amd/mhgp.py).

A user's program holds host point clouds (numpy arrays) and keeps a Context
(or a Server) for them; one pass of a case is one use of it:

  index      upload a cloud and read back its canonical points and LBVH
  emst       upload a cloud and compute its exact minimum spanning tree
  knn        exact neighbour lists of every point of an uploaded cloud
  partition  exact top-k partitions of rational query points
  ball       closed-ball partitions of supports of an uploaded cloud
  catalogue  upload a cloud and read back its critical-sphere catalogue
  pipeline   upload, spanning tree, catalogue and hgp_reduced tower, the tower
             read back (the warm end-to-end step of bench.py)
  serve      several clouds at once through the continuous-batching server
"""

from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
for _p in (ROOT, os.path.join(ROOT, "e-hgp_amd")):
    if _p not in sys.path:
        sys.path.insert(0, _p)

import mhgp  # noqa: E402
import workloads  # noqa: E402


def listed():
    return [
        # the smallest call: a cloud of the CPU-reference size indexed, where launches and waits count
        {"name": "index_256", "do": "index", "cloud": "uniform", "n": 256},
        # the largest cloud of the repository's configurations: snapped anisotropic blobs with noise
        {"name": "index_200k", "do": "index", "cloud": "snapped", "n": 200_000},
        # a spanning tree alone (single-linkage users), an odd size of unevenly dense blobs
        {"name": "emst_60001", "do": "emst", "cloud": "mixture", "n": 60_001},
        # the largest neighbour lists, on the cloud of the headline benchmark
        {"name": "knn_50k_k32", "do": "knn", "cloud": "lattice", "n": 50_000, "k": 32},
        # proposals for facet centres: rational queries, a few exclusions each
        {"name": "partition_20011", "do": "partition", "cloud": "lattice", "n": 20_011, "queries": 509, "k": 10},
        # spheres of 1..4 support points settled against the whole cloud
        {"name": "ball_50k", "do": "ball", "cloud": "lattice", "n": 50_000, "queries": 4_099, "cap": 16},
        # the smallest catalogue (256 uniform points, K_max 3), where latency counts
        {"name": "catalogue_256_k3", "do": "catalogue", "cloud": "uniform", "cloud_seed": 0, "n": 256, "k": 3},
        # every record of an anisotropic mixture, whose sparse points gather most of the cloud
        {"name": "catalogue_mixture_2003", "do": "catalogue", "cloud": "mixture", "cloud_seed": 4, "n": 2_003, "k": 10},
        # the smallest cloud of the batch workload, end to end
        {"name": "pipeline_1k_k10", "do": "pipeline", "cloud": "lattice", "cloud_seed": 0, "n": 1_000, "k": 10},
        # an ordinary cloud of the served stream at its smaller K_max
        {"name": "pipeline_17117_k4", "do": "pipeline", "cloud": "lattice", "cloud_seed": 0, "n": 17_117, "k": 4},
        # the headline benchmark's step
        {"name": "pipeline_50k_k10", "do": "pipeline", "cloud": "lattice", "cloud_seed": 0, "n": 50_000, "k": 10},
        # the served stream: lattices and mixtures together, four slots, the benchmark's enumeration budget
        {"name": "serve_6", "do": "serve", "cloud": "batch", "cloud_seed": 2, "n": 4_000, "clouds": 6, "slots": 4, "k": 10},
    ]


def draw(rng):
    def size(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    do = rng.choice(["index", "emst", "knn", "partition", "ball", "catalogue", "pipeline", "pipeline", "serve"])
    if do == "index":
        return {"do": do, "cloud": rng.choice(["uniform", "lattice", "mixture", "snapped"]), "n": size(64, 200_000)}
    if do == "emst":
        return {"do": do, "cloud": rng.choice(["uniform", "lattice", "mixture"]), "n": size(64, 60_001)}
    if do == "knn":
        return {"do": do, "cloud": rng.choice(["uniform", "lattice", "mixture"]), "n": size(64, 50_000),
                "k": rng.randint(1, 32)}
    if do == "partition":
        return {"do": do, "cloud": rng.choice(["uniform", "lattice"]), "n": size(256, 20_011), "queries": size(1, 509),
                "k": rng.randint(1, 32)}
    if do == "ball":
        return {"do": do, "cloud": rng.choice(["uniform", "lattice"]), "n": size(256, 50_000), "queries": size(1, 4_099),
                "cap": rng.randint(0, 16)}
    if do == "catalogue":
        cloud = rng.choice(["uniform", "lattice", "mixture"])
        return {"do": do, "cloud": cloud, "cloud_seed": rng.randrange(1 << 20),
                "n": size(64, 1_000 if cloud == "mixture" else 6_000), "k": rng.randint(1, 10)}
    if do == "pipeline":
        cloud = rng.choice(["uniform", "lattice", "lattice"])
        return {"do": do, "cloud": cloud, "cloud_seed": rng.randrange(1 << 20),
                "n": size(64, 12_000 if cloud == "uniform" else 50_000), "k": rng.randint(1, 10)}
    return {"do": do, "cloud": "batch", "cloud_seed": rng.randrange(1 << 20), "n": size(1_000, 4_000),
            "clouds": rng.randint(1, 6), "slots": rng.randint(1, 4), "k": rng.choice([4, 10])}


def _cloud(kind, n, seed):
    if kind == "uniform":
        return workloads.uniform_cloud(n, seed=seed)
    if kind == "lattice":
        return workloads.jittered_lattice(n, side=max(2, math.ceil((n * 1.01) ** (1 / 3))), sigma=0.1, seed=seed)
    blobs = 5 + seed % 16
    if kind == "mixture":
        return workloads.gaussian_mixture(n, blobs=blobs, noise_fraction=0.15, box=10.0, snap_bits=None, seed=seed)
    if kind == "snapped":
        return workloads.gaussian_mixture(n, blobs=blobs, noise_fraction=0.15, box=10.0, snap_bits=12, seed=seed)
    raise ValueError(kind)


def _placed(points, seed):
    """The cloud in another place, size and orientation (a signed permutation
    of its axes): other coordinates and PointIds, the same number of critical
    spheres and tower nodes, so that results of different seeds have one shape."""
    rng = np.random.default_rng(seed)
    turned = points[:, rng.permutation(3)] * rng.choice([-1.0, 1.0], size=3)
    return turned * rng.uniform(0.5, 2.0) + rng.uniform(-1.0, 1.0, size=3) * np.ptp(points)


def _queries(case, seed):
    """Rational query points (numerators over one denominator) in the cloud's
    box and 0..3 excluded PointIds per query."""
    rng = np.random.default_rng(seed + 77)
    pts = _cloud(case["cloud"], case["n"], seed)
    q = case["queries"]
    den = rng.integers(2, 1 << 12, size=q)
    spacing = (pts.max() - pts.min()) / len(pts) ** (1 / 3)
    at = pts[rng.integers(0, len(pts), size=q)] + rng.normal(0.0, 0.3, size=(q, 3)) * spacing
    num = np.rint(at * den[:, None]).astype(np.int64)
    excl = [sorted(int(x) for x in rng.choice(case["n"], size=int(m), replace=False)) for m in rng.integers(0, 4, size=q)]
    return pts, num, den, excl


def _points(case, seed):
    if "cloud_seed" in case:
        return _placed(_cloud(case["cloud"], case["n"], case["cloud_seed"]), seed)
    return _cloud(case["cloud"], case["n"], seed)


def prepare(case, seed):
    do = case["do"]
    if do == "serve":
        rng = np.random.default_rng(case["cloud_seed"])
        # sizes spread around n as the batch workload spreads them, half lattices, half mixtures
        sizes = np.exp(rng.uniform(np.log(0.5), np.log(1.5), size=case["clouds"])) * case["n"]
        clouds = []
        for i, m in enumerate(sizes):
            kind = "lattice" if (i + case["cloud_seed"]) % 2 else "mixture"
            clouds.append(_placed(_cloud(kind, int(m), case["cloud_seed"] * 31 + i), seed))
        return {"case": case, "clouds": clouds, "server": mhgp.Server(0, slots=case["slots"], region_limit=640)}
    ctx = mhgp.Context(0)
    state = {"case": case, "ctx": ctx}
    if do == "partition":
        state["points"], state["num"], state["den"], state["excl"] = _queries(case, seed)
        ctx.upload(state["points"])
        return state
    state["points"] = _points(case, seed)
    if do in ("knn", "ball"):
        ctx.upload(state["points"])
    if do == "ball":
        # supports as the streams propose them: a point and some of its nearest neighbours
        rng = np.random.default_rng(seed + 5)
        near = ctx.knn(12)
        anchors = rng.integers(0, case["n"], size=case["queries"])
        sup = []
        for u, m in zip(anchors, rng.integers(1, 5, size=case["queries"])):
            other = near[u][rng.choice(12, size=int(m) - 1, replace=False)]
            sup.append([int(u)] + [int(x) for x in other])
        state["supports"] = sup
    return state


def _tower(tw):
    return {k: tw[k] for k in ("order", "kind", "level_class", "level", "child_offset", "children", "vertical") if k in tw}


def run(state):
    case = state["case"]
    do = case["do"]
    if do == "serve":
        srv = state["server"]
        tickets = [srv.submit(p, case["k"]) for p in state["clouds"]]
        ends, towers = [], []
        for t in tickets:
            r = srv.wait(t)
            ends.append((r.code, r.status, r.event_count, r.node_count, r.child_count))
            if r.code == 0 and r.status == 0:
                towers.append(_tower(srv.fetch(t, r)))
            srv.release(t)
        return {"ends": np.asarray(ends, dtype=np.int64), "towers": towers}
    ctx = state["ctx"]
    if do == "index":
        ctx.upload(state["points"])
        xyz, source = ctx.canonical_points()
        leaves, nodes, counters = ctx.lbvh_snapshot()
        return {"xyz": xyz, "source": source, "leaves": leaves, "nodes": nodes, "counters": counters}
    if do == "emst":
        ctx.upload(state["points"])
        return {"edges": ctx.emst()}
    if do == "knn":
        return {"ids": ctx.knn(case["k"])}
    if do == "partition":
        parts = ctx.knn_partition(state["num"], state["den"], case["k"], exclusions=state["excl"])
        return {"cutoff_sq": np.array([p["cutoff_sq"] for p in parts]),
                "cutoff_id": np.array([p["cutoff_id"] for p in parts]),
                "choice": np.array([p["choice"] for p in parts]),
                "strict": np.array([x for p in parts for x in p["strict"]], dtype=np.int64),
                "strict_count": np.array([len(p["strict"]) for p in parts]),
                "shell": np.array([x for p in parts for x in p["shell"]], dtype=np.int64),
                "shell_count": np.array([p["shell_count"] for p in parts])}
    if do == "ball":
        inter, nin, nsh = ctx.closed_ball(state["supports"], cap=case["cap"])
        return {"interior": inter, "interior_count": nin, "shell_count": nsh}
    if do == "catalogue":
        ctx.upload(state["points"])
        cat = ctx.supports_raw(case["k"])
        return {k: cat[k] for k in ("ids", "meta", "interior", "level", "level_class")}
    ctx.upload(state["points"])
    edges = ctx.emst()
    info = ctx.supports(case["k"], fetch=False)
    out = {"edges": edges, "events": info.event_count, "diagnostics": info.diagnostic_count}
    if info.status == 0 and info.diagnostic_count == 0:
        out["tower"] = _tower(ctx.tower(case["k"], fetch=True))
    return out


def work(case):
    do, n = case["do"], case["n"]
    cloud = 24 * n  # binary64 coordinates in
    if do == "index":
        # out: canonical coordinates, source indices, leaves (16 B), 2n - 1 nodes of 80 B; three key sorts' comparisons
        return {"bytes": cloud + n * (24 + 4 + 16 + 160), "flops": n * 4 * math.log2(n + 1)}
    if do == "emst":
        return {"bytes": cloud + 8 * n, "flops": 8 * n * math.log2(n + 1)}
    if do == "knn":
        # every listed distance evaluated once (8 operations)
        return {"bytes": cloud + 4 * n * case["k"], "flops": 8 * n * case["k"]}
    if do == "partition":
        q = case["queries"]
        return {"bytes": min(cloud, q * case["k"] * 24 * 4) + q * (32 + 12 * case["k"] + 20), "flops": 8 * q * case["k"]}
    if do == "ball":
        q = case["queries"]
        return {"bytes": min(cloud, q * 24 * 16) + q * (17 + 4 * case["cap"] + 8), "flops": 150 * q}
    # records and tower nodes of a generic cloud grow about so per point
    k = case["k"]
    records, nodes = n * (0.45 * k**3 + 4 * k), n * (0.45 * k * k + 1)
    # each record: its sphere (about 100 operations) and its closed ball's points tested once (20 each)
    flops = records * (100 + 20 * (k + 1))
    if do == "catalogue":
        return {"bytes": cloud + records * (16 + 4 + 4 * k + 8 + 8), "flops": flops}
    tower = nodes * (4 + 4 + 8 + 8 + 8 + 8 + 8)
    if do == "pipeline":
        return {"bytes": cloud + 8 * n + tower, "flops": flops}
    return {"bytes": case["clouds"] * (cloud + tower), "flops": case["clouds"] * flops}


def _exact_levels(points, k_max):
    """Squared radii of every critical sphere of closed rank <= k_max + 1, by
    exhaustive search over supports of 2..4 points, ascending."""
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    p = torch.tensor(points, dtype=torch.float64, device=dev)
    n = len(p)
    s_max = min(min(k_max, n) + 1, n)
    levels = []

    def keep(center, r2, m):
        for c, r in zip(center.split(1 << 18), r2.split(1 << 18)):
            d2 = torch.zeros((len(c), n), dtype=torch.float64, device=dev)
            for a in range(3):
                d2 += (p[None, :, a] - c[:, a, None]) ** 2
            inside = (d2 < r[:, None] * (1 - 1e-9)).sum(1)
            levels.append(r[inside + m <= s_max])

    def dot(a, b):
        return (a * b).sum(-1)

    i, j = torch.triu_indices(n, n, 1, device=dev)
    keep((p[i] + p[j]) / 2, dot(p[i] - p[j], p[i] - p[j]) / 4, 2)
    if s_max >= 3:
        for u in range(n - 2):
            a, b = torch.triu_indices(n - u - 1, n - u - 1, 1, device=dev) + u + 1
            v, w = p[a] - p[u], p[b] - p[u]
            vv, ww, vw = dot(v, v), dot(w, w), dot(v, w)
            det = 2 * (vv * ww - vw * vw)
            s, t = ww * (vv - vw) / det, vv * (ww - vw) / det
            ok = (s > 0) & (t > 0) & (s + t < 1)
            off = s[:, None] * v + t[:, None] * w
            keep((off + p[u])[ok], dot(off, off)[ok], 3)
            if s_max < 4 or u >= n - 3:
                continue
            # tetrahedra (u, a < b < z): barycentric coordinates of the circumcentre all positive
            for part in range(0, len(a), 16384):
                av, bv = a[part : part + 16384], b[part : part + 16384]
                rows, z = torch.nonzero(torch.arange(n, device=dev)[None, :] > bv[:, None], as_tuple=True)
                if not len(rows):
                    continue
                v, w, x = p[av[rows]] - p[u], p[bv[rows]] - p[u], p[z] - p[u]
                vxw, wxx, xxv = torch.linalg.cross(v, w), torch.linalg.cross(w, x), torch.linalg.cross(x, v)
                vol = 2 * dot(v, wxx)
                off = (dot(v, v)[:, None] * wxx + dot(w, w)[:, None] * xxv + dot(x, x)[:, None] * vxw) / vol[:, None]
                la, lb, lc = 2 * dot(off, wxx) / vol, 2 * dot(off, xxv) / vol, 2 * dot(off, vxw) / vol
                ok = (la > 0) & (lb > 0) & (lc > 0) & (la + lb + lc < 1)
                keep((off + p[u])[ok], dot(off, off)[ok], 4)
    return torch.sort(torch.cat(levels)).values.cpu().numpy()


def exact(case, seed):
    do = case["do"]
    if do == "index":
        pts = _cloud(case["cloud"], case["n"], seed) + 0.0
        order = np.lexsort((pts[:, 2], pts[:, 1], pts[:, 0]))
        return {"xyz": pts[order], "source": None, "leaves": None, "nodes": None, "counters": None}
    if do == "partition":
        pts, num, den, excl = _queries(case, seed)
        canon = pts[np.lexsort((pts[:, 2], pts[:, 1], pts[:, 0]))].astype(np.longdouble)
        cut = []
        for q in range(len(num)):
            d = ((canon - num[q].astype(np.longdouble) / np.longdouble(den[q])) ** 2).sum(1)
            d[excl[q]] = np.inf
            cut.append(float(np.partition(d, case["k"] - 1)[case["k"] - 1]))
        return {"cutoff_sq": np.array(cut), "cutoff_id": None, "choice": None, "strict": None, "strict_count": None,
                "shell": None, "shell_count": None}
    if do == "catalogue" and case["n"] <= 256:
        levels = _exact_levels(_points(case, seed), case["k"])
        return {"ids": None, "meta": None, "interior": None, "level": levels, "level_class": None}
    return None
