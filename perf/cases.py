"""Performance cases of the BVH query and mesh sampling path: what users of the library have it do,
through its public entry points, from batches of a few dozen queries to 10 million.

Inputs are synthetic and seeded: noise-displaced tori and perturbed spheres (single scans or
models), scenes of 64 ellipsoids, and queries uniform in the inflated bounding box or near the
surface. Results of the library are canonical (lowest index on exact ties) and bit-exact whatever
tree or traversal order is used, so index, distance and hit outputs are compared exactly; only the
ICP transforms, sums of many doubles, carry a tolerance.
"""
import math

import numpy as np
import torch

import thea_amd
from thea_amd.batch import BatchPlan
from thea_amd.serve import Server

DEV = "cuda:0"


# ---- listed and drawn cases ----------------------------------------------------------------------
def listed():
    return [
        # a tool probing a model a few points at a time: launch and walk latency only
        dict(name="closest_few", kind="closest", shape="sphere", tris=20_480, n=61, leaf=4, where="near", bound=-1.0),
        # a sparse, bounded probe of a large scan (snapping markers to a surface)
        dict(name="closest_sparse", kind="closest", shape="torus", tris=1_048_576, n=3_001, leaf=4, where="box",
             bound=0.5),
        # an ordinary model and point cloud (the 20,480-triangle sphere, 100,000 queries)
        dict(name="closest_mid", kind="closest", shape="sphere", tris=20_480, n=100_000, leaf=4, where="box",
             bound=-1.0),
        # the headline: a million triangles, ten million queries filling the box
        dict(name="closest_large", kind="closest", shape="torus", tris=1_048_576, n=10_000_000, leaf=12, where="box",
             bound=-1.0),
        # neighbourhood graph of a sampled scene: each point's nearest others
        dict(name="knn_points", kind="knn", points=1_000_003, k=16, leaf=16, exclude=True),
        # ray casting: random first hits with normals
        dict(name="rays_first", kind="rays", shape="torus", tris=1_048_576, n=4_000_000, leaf=2),
        # shadow/occlusion rays of limited length from surface points
        dict(name="rays_any", kind="occlusion", shape="torus", tris=250_000, n=2_000_001, leaf=1, reach=0.7),
        # area-weighted surface samples of the 128,000-triangle ellipsoid scene
        dict(name="sample_area", kind="sample", ellipsoids=64, n=1_000_000),
        # a mesh that changes each frame: upload, build, query
        dict(name="build_query", kind="build", shape="torus", tris=999_698, n=200_000, leaf=8),
        # many meshes of uneven size, built and queried by one plan
        dict(name="batch_many", kind="batch", meshes=96, tri_max=120_000, query_max=60_000),
        # mixed requests on resident meshes: 60% closest point, 25% 8-NN, 15% rays
        dict(name="serve_mix", kind="serve", meshes=12, tri_max=700_000, requests=60, size_max=200_000),
        # rotation search of scan alignment: 24 starts, host arrays in and out, double target
        dict(name="icp_search", kind="icp", n=60_000, target=80_000, starts=24, iterations=4),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["closest", "closest", "closest", "knn", "rays", "occlusion", "sample", "build", "batch",
                       "serve", "icp"])
    shape = rng.choice(["torus", "sphere"])
    tris = _logint(rng, 2_000, 1_048_576)
    if kind == "closest":
        n = _logint(rng, 32, 8_000_000)
        return dict(kind=kind, shape=shape, tris=tris if shape == "torus" or n < 300_000 else min(tris, 100_000), n=n,
                    leaf=rng.choice([4, 4, 8, 12]), where=rng.choice(["box", "near"]) if shape == "torus" else "near",
                    bound=rng.choice([-1.0, -1.0, 0.3]))
    if kind == "knn":
        return dict(kind=kind, points=_logint(rng, 5_000, 1_500_000), k=rng.choice([1, 3, 8, 10, 16]),
                    leaf=rng.choice([4, 16]), exclude=rng.choice([True, False]))
    if kind == "rays":
        return dict(kind=kind, shape=shape, tris=tris, n=_logint(rng, 100, 6_000_000), leaf=rng.choice([1, 2, 4]))
    if kind == "occlusion":
        return dict(kind=kind, shape=shape, tris=tris, n=_logint(rng, 100, 6_000_000), leaf=rng.choice([1, 2, 4]),
                    reach=rng.choice([0.2, 0.7, 2.0]))
    if kind == "sample":
        return dict(kind=kind, ellipsoids=_logint(rng, 2, 128), n=_logint(rng, 1_000, 4_000_000))
    if kind == "build":
        return dict(kind=kind, shape=shape, tris=tris, n=_logint(rng, 100, 300_000), leaf=rng.choice([4, 8]))
    if kind == "batch":
        return dict(kind=kind, meshes=_logint(rng, 4, 128), tri_max=_logint(rng, 5_000, 120_000),
                    query_max=_logint(rng, 2_000, 60_000))
    if kind == "serve":
        return dict(kind=kind, meshes=rng.randint(2, 12), tri_max=_logint(rng, 30_000, 700_000),
                    requests=rng.randint(10, 60), size_max=_logint(rng, 2_000, 200_000))
    return dict(kind=kind, n=_logint(rng, 1_000, 80_000), target=_logint(rng, 1_000, 80_000),
                starts=rng.choice([1, 6, 24]), iterations=4)


# ---- inputs --------------------------------------------------------------------------------------
def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((int(seed) * 1_000_003 + stream) & 0x7FFFFFFF)
    return g


def _rand(g, *shape):
    return torch.rand(*shape, generator=g, device=DEV, dtype=torch.float64)


def _grid_faces(nu, nv):
    """Two triangles per cell of a periodic nu x nv grid."""
    i = torch.arange(nu, device=DEV)[:, None]
    j = torch.arange(nv, device=DEV)[None, :]
    i1, j1 = (i + 1) % nu, (j + 1) % nv
    a, b, c, d = i * nv + j, i1 * nv + j, i1 * nv + j1, i * nv + j1
    return torch.stack([torch.stack([a, b, c], -1), torch.stack([a, c, d], -1)], 2).reshape(-1, 3).to(torch.int32)


def _torus(tris, g):
    """Torus R = 1, r = 0.3, its minor radius displaced by smooth periodic noise of amplitude 0.05."""
    nv = max(3, int(round(math.sqrt(tris / 4))))
    nu = max(3, int(round(tris / (2 * nv))))
    u = 2 * math.pi * torch.arange(nu, device=DEV, dtype=torch.float64)[:, None] / nu
    w = 2 * math.pi * torch.arange(nv, device=DEV, dtype=torch.float64)[None, :] / nv
    amp, ph = _rand(g, 12) - 0.5, 2 * math.pi * _rand(g, 12)
    noise = torch.zeros(nu, nv, device=DEV, dtype=torch.float64)
    for k in range(12):
        noise += amp[k] * torch.sin((3 + 2 * k) * u + (1 + k) * w + ph[k])
    r = 0.3 + 0.05 * noise / noise.abs().max()
    x, y, z = (1 + r * torch.cos(w)) * torch.cos(u), (1 + r * torch.cos(w)) * torch.sin(u), r * torch.sin(w)
    return torch.stack([x, y, z], -1).reshape(-1, 3).to(torch.float32), _grid_faces(nu, nv)


def _uv_sphere(tris):
    """Unit sphere of about `tris` triangles: rings of latitude and two poles."""
    rings = max(3, int(round(math.sqrt(tris / 4))))
    slices = max(3, int(round(tris / (2 * rings))))
    th = math.pi * (torch.arange(rings, device=DEV, dtype=torch.float64)[:, None] + 1) / (rings + 1)
    ph = 2 * math.pi * torch.arange(slices, device=DEV, dtype=torch.float64)[None, :] / slices
    ring = torch.stack([torch.sin(th) * torch.cos(ph), torch.sin(th) * torch.sin(ph),
                        torch.cos(th).expand(rings, slices)], -1).reshape(-1, 3)
    poles = torch.tensor([[0.0, 0.0, 1.0], [0.0, 0.0, -1.0]], device=DEV, dtype=torch.float64)
    v = torch.cat([ring, poles])
    i = torch.arange(rings - 1, device=DEV)[:, None]
    j = torch.arange(slices, device=DEV)[None, :]
    j1 = (j + 1) % slices
    a, b, c, d = i * slices + j, (i + 1) * slices + j, (i + 1) * slices + j1, i * slices + j1
    mid = torch.stack([torch.stack([a, b, c], -1), torch.stack([a, c, d], -1)], 2).reshape(-1, 3)
    top, bot = rings * slices, rings * slices + 1
    j, j1 = j[0], j1[0]
    base = (rings - 1) * slices
    caps = torch.cat([torch.stack([torch.full_like(j, top), j, j1], -1),
                      torch.stack([torch.full_like(j, bot), base + j1, base + j], -1)])
    return v, torch.cat([mid, caps]).to(torch.int32)


def _mesh(shape, tris, g):
    if shape == "torus":
        return _torus(tris, g)
    v, t = _uv_sphere(tris)  # vertex radii perturbed by N(0, 0.02)
    s = 1 + 0.02 * torch.randn(len(v), 1, generator=g, device=DEV, dtype=torch.float64)
    return (v * s).to(torch.float32), t


def _ellipsoids(count, g):
    """Union of `count` ellipsoids of 2,000 triangles, semi-axes U[0.05, 0.3], centres U[-1, 1]^3."""
    v, t = _uv_sphere(2_000)
    ax, c = 0.05 + 0.25 * _rand(g, count, 1, 3), 2 * _rand(g, count, 1, 3) - 1
    off = torch.arange(count, device=DEV, dtype=torch.int32)[:, None, None] * len(v)
    return (v[None] * ax + c).reshape(-1, 3).to(torch.float32), (t[None] + off).reshape(-1, 3).contiguous()


def _box_points(v, n, g):
    """Uniform in the bounding box inflated 20%."""
    lo, hi = v.min(0).values.double(), v.max(0).values.double()
    c, h = (lo + hi) / 2, 0.6 * (hi - lo)
    return (c + h * (2 * _rand(g, n, 3) - 1)).to(torch.float32)


def _near_points(v, t, n, g, spread=0.01):
    """Scan-like points: on random triangles, moved by Gaussian noise."""
    f = t[torch.randint(len(t), (n,), generator=g, device=DEV)].long()
    a, b = _rand(g, n, 1), _rand(g, n, 1)
    s = torch.sqrt(a)
    p = (1 - s) * v[f[:, 0]].double() + s * (1 - b) * v[f[:, 1]].double() + s * b * v[f[:, 2]].double()
    return (p + spread * torch.randn(n, 3, generator=g, device=DEV, dtype=torch.float64)).to(torch.float32)


def _directions(n, g):
    d = torch.randn(n, 3, generator=g, device=DEV, dtype=torch.float64)
    return (d / d.norm(dim=1, keepdim=True)).to(torch.float32)


def _spread_sizes(lo, hi, count):
    """`count` sizes evenly spaced in their logarithm, in a mixed order."""
    f = [((i * 0.6180339887498949) % 1.0) for i in range(count)]
    return [int(round(lo * (hi / lo) ** x)) for x in f]


def _rotations(starts):
    """`starts` rotations about the vertical axis and a tilt, as (K, 3, 4) transforms."""
    out = np.zeros((starts, 3, 4))
    for i in range(starts):
        a, b = 2 * math.pi * i / max(starts, 1), 0.4 * (i % 3)
        rz = np.array([[math.cos(a), -math.sin(a), 0], [math.sin(a), math.cos(a), 0], [0, 0, 1]])
        rx = np.array([[1, 0, 0], [0, math.cos(b), -math.sin(b)], [0, math.sin(b), math.cos(b)]])
        out[i, :, :3] = rz @ rx
    return out


def _closest_inputs(case, seed):
    g = _gen(seed, 1)
    v, t = _mesh(case["shape"], case["tris"], g)
    q = _box_points(v, case["n"], g) if case["where"] == "box" else _near_points(v, t, case["n"], g)
    return v, t, q


def _knn_inputs(case, seed):
    g = _gen(seed, 2)
    v, t = _ellipsoids(64, g)
    return _near_points(v, t, case["points"], g, spread=1e-4)


def _ray_inputs(case, seed):
    g = _gen(seed, 3)
    v, t = _mesh(case["shape"], case["tris"], g)
    if case["kind"] == "rays":
        return v, t, _box_points(v, case["n"], g), _directions(case["n"], g)
    d = _directions(case["n"], g)
    o = _near_points(v, t, case["n"], g, spread=0.0).double() + 0.02 * d.double()
    return v, t, o.to(torch.float32), d


def _batch_inputs(case, seed):
    g = _gen(seed, 4)
    verts, tris, queries = [], [], []
    nt = _spread_sizes(1_000, case["tri_max"], case["meshes"])
    nq = _spread_sizes(1_000, case["query_max"], case["meshes"] + 7)[7:]
    for m in range(case["meshes"]):
        v, t = _mesh("torus" if m % 2 else "sphere", nt[m], g)
        v = (v.double() * (0.5 + 1.5 * _rand(g, 1)) + 20 * _rand(g, 1, 3) - 10).to(torch.float32)
        verts.append(v)
        tris.append(t)
        queries.append(_box_points(v, nq[m], g))
    return verts, tris, queries


def _serve_inputs(case, seed):
    g = _gen(seed, 5)
    sizes = _spread_sizes(10_000, case["tri_max"], case["meshes"])
    meshes = [_mesh("torus" if m % 2 else "sphere", s, g) for m, s in enumerate(sizes)]
    ns = _spread_sizes(256, case["size_max"], case["requests"])
    reqs = []
    for i, n in enumerate(ns):
        m = (i * 5) % case["meshes"]
        kind = ("closest", "knn", "closest", "ray", "closest", "closest", "knn", "closest", "knn", "closest",
                "ray", "closest", "closest", "knn", "closest", "closest", "ray", "closest", "knn", "closest")[i % 20]
        q = _box_points(meshes[m][0], n, g)
        reqs.append((kind, m, q, _directions(n, g) if kind == "ray" else None))
    return meshes, reqs


def _icp_inputs(case, seed):
    g = _gen(seed, 6)
    v, t = _torus(100_000, g)
    target = _near_points(v, t, case["target"], g, 0.0).double().cpu().numpy()
    src = _near_points(v, t, case["n"], g, 0.002).double().cpu().numpy()
    a = 0.15
    r = np.array([[math.cos(a), -math.sin(a), 0], [math.sin(a), math.cos(a), 0], [0, 0, 1]])
    return np.ascontiguousarray(src @ r.T + np.array([0.02, -0.01, 0.015])), np.ascontiguousarray(target)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "closest":
        v, t, q = _closest_inputs(case, seed)
        mesh = thea_amd.Mesh(v, t)
        state = dict(bvh=thea_amd.MeshBvh(mesh, leaf_size=case["leaf"]), q=q)
    elif kind == "knn":
        p = _knn_inputs(case, seed)
        state = dict(bvh=thea_amd.PointBvh(p, leaf_size=case["leaf"]), q=p)
    elif kind in ("rays", "occlusion"):
        v, t, o, d = _ray_inputs(case, seed)
        state = dict(bvh=thea_amd.MeshBvh(thea_amd.Mesh(v, t), leaf_size=case["leaf"]), o=o, d=d)
    elif kind == "sample":
        v, t = _ellipsoids(case["ellipsoids"], _gen(seed, 7))
        mesh = thea_amd.Mesh(v, t)
        mesh.total_area()  # the area distribution is made once per mesh
        state = dict(sampler=thea_amd.MeshSampler(mesh), seed=seed & 0xFFFF)
    elif kind == "build":
        g = _gen(seed, 8)
        v, t = _mesh(case["shape"], case["tris"], g)
        state = dict(v=v, t=t, q=_near_points(v, t, case["n"], g))
    elif kind == "batch":
        verts, tris, queries = _batch_inputs(case, seed)
        plan = BatchPlan([len(x) for x in verts], [len(x) for x in tris], [len(x) for x in queries])
        state = dict(plan=plan, v=torch.cat(verts), t=torch.cat(tris), q=torch.cat(queries))
    elif kind == "serve":
        meshes, reqs = _serve_inputs(case, seed)
        server = Server()
        ids = [server.add_mesh(v.cpu().numpy(), t.cpu().numpy()) for v, t in meshes]
        totals = {}
        for k, _, q, _ in reqs:
            totals[k] = totals.get(k, 0) + len(q)
        state = dict(server=server, reqs=[(k, ids[m], q, d) for k, m, q, d in reqs], totals=totals)
    else:
        src, target = _icp_inputs(case, seed)
        icp = thea_amd.Icp3(-1.0, case["iterations"], case["iterations"], kabsch=True)
        state = dict(icp=icp, src=src, bvh=thea_amd.PointBvhF64(target), init=_rotations(case["starts"]))
    torch.cuda.synchronize()
    state["case"] = case
    return state


# ---- one pass ------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "closest":
        return state["bvh"].closestPoint(state["q"], case["bound"])
    if kind == "knn":
        return state["bvh"].kClosestElements(state["q"], case["k"], exclude_self=case["exclude"])
    if kind == "rays":
        return state["bvh"].rayStructureIntersection(state["o"], state["d"])
    if kind == "occlusion":
        return state["bvh"].rayIntersects(state["o"], state["d"], case["reach"])
    if kind == "sample":
        return state["sampler"].sampleEvenlyByArea(case["n"], seed=state["seed"], device=True)
    if kind == "build":
        bvh = thea_amd.MeshBvh(thea_amd.Mesh(state["v"], state["t"]), leaf_size=case["leaf"])
        return bvh.closestPoint(state["q"])
    if kind == "batch":
        return state["plan"].run(state["v"], state["t"], state["q"])
    if kind == "serve":
        server, pending, outs, used = state["server"], [], {}, {}
        for k, n in state["totals"].items():  # one result buffer per kind, a slice of it per request
            cols = 8 if k == "knn" else 1
            outs[k] = dict(idx=torch.empty(n, cols, dtype=torch.int32, device=DEV),
                           dist=torch.empty(n, cols, dtype=torch.float32, device=DEV),
                           cp=None if k == "knn" else torch.empty(n, 3, dtype=torch.float32, device=DEV))
        for k, m, q, d in state["reqs"]:
            a = used.get(k, 0)
            used[k] = b = a + len(q)
            o = {key: None if x is None else x[a:b] for key, x in outs[k].items()}
            rid, _ = server.submit(k, m, q, dirs=d, k=8 if k == "knn" else 0, outputs=o)
            pending.append(rid)
        for rid in pending:
            rc, _ = server.wait(rid)
            if rc != 0:
                raise RuntimeError(f"request {rid} ended with status {rc}")
        return [x for k in sorted(outs) for x in outs[k].values() if x is not None]
    return state["icp"].alignBatch(state["src"], state["bvh"], state["init"])


# ---- what a pass cannot do without ---------------------------------------------------------------
def _walk_flops(n, elements, per_element):
    """A descent by halving (two box distances, 30 operations, per level) and one exact element."""
    return n * (30.0 * math.log2(max(elements, 2)) + per_element)


def work(case):
    kind = case["kind"]
    tri_bytes = 18.0  # a closed mesh: 12 bytes of indices and half a 12-byte vertex per triangle
    if kind == "closest":
        return dict(bytes=case["n"] * 32.0 + case["tris"] * tri_bytes, flops=_walk_flops(case["n"], case["tris"], 80))
    if kind == "knn":
        n, k = case["points"], case["k"]
        return dict(bytes=n * (12.0 + 8.0 * k) + 12.0 * n, flops=_walk_flops(n, n, 8 * k))
    if kind == "rays":
        return dict(bytes=case["n"] * (24.0 + 20.0) + case["tris"] * tri_bytes,
                    flops=_walk_flops(case["n"], case["tris"], 50))
    if kind == "occlusion":
        return dict(bytes=case["n"] * 25.0 + case["tris"] * tri_bytes, flops=_walk_flops(case["n"], case["tris"], 50))
    if kind == "sample":
        t = 2_000.0 * case["ellipsoids"]
        return dict(bytes=case["n"] * 28.0 + t * (tri_bytes + 8.0), flops=case["n"] * (80 + math.log2(t)))
    if kind == "build":
        return dict(bytes=case["tris"] * tri_bytes + case["n"] * 32.0,
                    flops=case["tris"] * 100.0 + _walk_flops(case["n"], case["tris"], 80))
    if kind == "batch":
        nt = _spread_sizes(1_000, case["tri_max"], case["meshes"])
        nq = _spread_sizes(1_000, case["query_max"], case["meshes"] + 7)[7:]
        return dict(bytes=sum(nt) * tri_bytes + sum(nq) * 20.0,
                    flops=sum(nt) * 100.0 + sum(_walk_flops(q, t, 80) for q, t in zip(nq, nt)))
    if kind == "serve":
        n = sum(_spread_sizes(256, case["size_max"], case["requests"]))
        t = sum(_spread_sizes(10_000, case["tri_max"], case["meshes"]))
        return dict(bytes=n * 45.0 + t * tri_bytes, flops=_walk_flops(n, t / case["meshes"], 150))
    visits = case["n"] * case["starts"] * (case["iterations"] + 1.0)
    return dict(bytes=case["n"] * 24.0 + case["target"] * 24.0 + visits * 24.0,
                flops=_walk_flops(visits, case["target"], 60))


def tolerance(case):
    # Every index, distance, point and hit is the canonical minimum of fixed float arithmetic.
    # ICP sums n doubles for the means, the covariance and the error: other summation orders move a
    # transform by some ulps (2e-15 relative against the 64-bit loop below, 1,000 to 80,000 points).
    return {"rel": 1e-14} if case["kind"] == "icp" else "exact"


# ---- 64-bit references ---------------------------------------------------------------------------
def _dot(a, b):
    return (a * b).sum(-1)


def _tri_closest64(p, a, b, c):
    """Squared distance and closest point of points p (n, 1, 3) to triangles (1, m, 3)."""
    def seg(o, d):
        s = (_dot(p - o, d) / _dot(d, d).clamp_min(1e-300)).clamp(0, 1)
        x = o + s[..., None] * d
        return _dot(p - x, p - x), x

    ab, ac = b - a, c - a
    nrm = torch.linalg.cross(ab, ac)
    n2 = _dot(nrm, nrm).clamp_min(1e-300)
    ap = p - a
    v = _dot(torch.linalg.cross(ap, ac.expand_as(ap)), nrm) / n2
    w = _dot(torch.linalg.cross(ab.expand_as(ap), ap), nrm) / n2
    inside = (v >= 0) & (w >= 0) & (v + w <= 1)
    h = _dot(ap, nrm) / n2
    best, x = seg(a, ab)
    for o, d in ((b, c - b), (c, a - c)):
        d2, y = seg(o, d)
        x = torch.where((d2 < best)[..., None], y, x)
        best = torch.minimum(d2, best)
    x = torch.where(inside[..., None], p - h[..., None] * nrm, x)
    return torch.where(inside, h * h * n2, best), x


def _closest64(v, t, q, bound):
    v64, q64 = v.double(), q.double()
    tri = v64[t.long()]
    best = torch.full((len(q),), math.inf, device=DEV, dtype=torch.float64)
    cp = torch.zeros(len(q), 3, device=DEV, dtype=torch.float64)
    step = 4096
    for i in range(0, len(q), step):
        p = q64[i:i + step]
        chunk = max(1, 4_000_000 // len(p))
        for j in range(0, len(tri), chunk):
            f = tri[j:j + chunk][None]
            d2, x = _tri_closest64(p[:, None], f[:, :, 0], f[:, :, 1], f[:, :, 2])
            m, k = d2.min(1)
            new = m < best[i:i + step]
            cp[i:i + step] = torch.where(new[:, None], x[torch.arange(len(p), device=DEV), k], cp[i:i + step])
            best[i:i + step] = torch.minimum(m, best[i:i + step])
    d = best.sqrt()
    if bound >= 0:
        none = d >= bound
        d = torch.where(none, torch.full_like(d, -1.0), d)
        cp = torch.where(none[:, None], torch.zeros_like(cp), cp)
    return d, cp


def _rays64(v, t, o, d, limit):
    """First hit times within [0, limit) (inf: none) and the unit normals of the hit faces."""
    tri = v.double()[t.long()]
    o64, d64 = o.double(), d.double()
    best = torch.full((len(o),), math.inf, device=DEV, dtype=torch.float64)
    which = torch.zeros(len(o), device=DEV, dtype=torch.long)
    a, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    face = torch.linalg.cross(e1, e2)
    step = 4096
    for i in range(0, len(o), step):
        p, r = o64[i:i + step, None], d64[i:i + step, None]
        chunk = max(1, 4_000_000 // len(p))
        for j in range(0, len(tri), chunk):
            n = face[None, j:j + chunk]
            den = -_dot(r, n)
            ap = p - a[None, j:j + chunk]
            q = torch.linalg.cross(ap, r.expand_as(ap))
            time = _dot(ap, n) / den
            u = _dot(e2[None, j:j + chunk], q) / den
            w = -_dot(e1[None, j:j + chunk], q) / den
            ok = (u >= 0) & (w >= 0) & (u + w <= 1) & (time >= 0) & (time < limit)
            m, k = torch.where(ok, time, torch.full_like(time, math.inf)).min(1)
            new = m < best[i:i + step]
            which[i:i + step] = torch.where(new, k + j, which[i:i + step])
            best[i:i + step] = torch.minimum(m, best[i:i + step])
    nrm = face[which] / face[which].norm(dim=1, keepdim=True).clamp_min(1e-300)
    return best, torch.where(torch.isinf(best)[:, None], torch.zeros_like(nrm), nrm)


def _philox(counter, key):
    """Philox4x32-10 (Salmon et al., SC 2011) at counters (counter, 0, 0, 0): (n, 4) words."""
    mask = np.uint64(0xFFFFFFFF)
    c = [counter.astype(np.uint64) & mask, counter.astype(np.uint64) >> np.uint64(32),
         np.zeros(len(counter), np.uint64), np.zeros(len(counter), np.uint64)]
    k = [key & 0xFFFFFFFF, key >> 32]
    for _ in range(10):
        p0, p1 = c[0] * np.uint64(0xD2511F53), c[2] * np.uint64(0xCD9E8D57)
        c = [(p1 >> np.uint64(32)) ^ c[1] ^ np.uint64(k[0]), p1 & mask,
             (p0 >> np.uint64(32)) ^ c[3] ^ np.uint64(k[1]), p0 & mask]
        k = [(k[0] + 0x9E3779B9) & 0xFFFFFFFF, (k[1] + 0xBB67AE85) & 0xFFFFFFFF]
    return np.stack(c, 1)


def _sample64(v, t, n, seed):
    v64, t = v.double().cpu().numpy(), t.cpu().numpy()
    a, e1, e2 = v64[t[:, 0]], v64[t[:, 1]] - v64[t[:, 0]], v64[t[:, 2]] - v64[t[:, 0]]
    cr = np.cross(e1, e2)
    len2 = np.linalg.norm(cr, axis=1)
    cdf = np.cumsum(0.5 * len2)
    u = _philox(np.arange(n), seed)[:, :3].astype(np.uint32).astype(np.float32) * np.float32(2.0 ** -32)
    tri = np.minimum(np.searchsorted(cdf, u[:, 0].astype(np.float64) * cdf[-1]), len(t) - 1)
    x, y = u[:, 1].astype(np.float64), u[:, 2].astype(np.float64)
    fold = x + y > 1
    x, y = np.where(fold, 1 - x, x), np.where(fold, 1 - y, y)
    pos = a[tri] + x[:, None] * e1[tri] + y[:, None] * e2[tri]
    return pos, (cr / np.maximum(len2, 1e-300)[:, None])[tri]


def _nearest64(p, target):
    out = torch.empty_like(p)
    step = max(1, 100_000_000 // (3 * len(target)))
    for i in range(0, len(p), step):
        d = p[i:i + step, None] - target[None]
        out[i:i + step] = target[(d * d).sum(-1).argmin(1)]
    return out


def _icp64(src, target, init, its):
    """The library's loop for a fixed number of iterations with least-squares rotations: each fit
    uses the correspondences of the positions before the previous update."""
    s0, tgt = torch.as_tensor(src, device=DEV), torch.as_tensor(target, device=DEV)
    trs, errs = [], []
    for m in torch.as_tensor(init, device=DEV):
        first = s0 @ m[:, :3].T + m[:, 3]
        pos, near = first, _nearest64(first, tgt)
        lin, off = torch.eye(3, device=DEV, dtype=torch.float64), torch.zeros(3, device=DEV, dtype=torch.float64)
        err = 0.0
        for _ in range(its):
            pm, qm = pos.mean(0), near.mean(0)
            u, _, vt = np.linalg.svd(((pos - pm).T @ (near - qm)).cpu().numpy())
            rot = torch.as_tensor((u @ vt).T.copy(), device=DEV)
            step = qm - rot @ pm
            lin, off = rot @ lin, rot @ off + step
            near = _nearest64(pos, tgt)
            pm, qm = pos.mean(0), near.mean(0)
            d = rot @ pm + step - qm
            r = (pos - pm) @ rot.T - (near - qm)
            err = float(d @ d) + float((r * r).sum())
            pos = first @ lin.T + off
        trs.append(np.hstack([lin.cpu().numpy(), off.cpu().numpy()[:, None]]))
        errs.append(err)
    return np.stack(trs), np.array(errs)


def exact(case, seed):
    kind = case["kind"]
    if kind == "closest":
        if float(case["n"]) * case["tris"] > 4e9:
            return None
        v, t, q = _closest_inputs(case, seed)
        d, cp = _closest64(v, t, q, case["bound"])
        return None, d, cp
    if kind == "build":
        if float(case["n"]) * case["tris"] > 4e9:
            return None
        g = _gen(seed, 8)
        v, t = _mesh(case["shape"], case["tris"], g)
        d, cp = _closest64(v, t, _near_points(v, t, case["n"], g), -1.0)
        return None, d, cp
    if kind == "knn":
        n = case["points"]
        if float(n) * n > 4e9:
            return None
        p = _knn_inputs(case, seed).double()
        out = torch.empty(n, case["k"], device=DEV, dtype=torch.float64)
        step = max(1, 50_000_000 // n)
        for i in range(0, n, step):
            e = p[i:i + step, None] - p[None]
            d2 = (e * e).sum(-1)
            if case["exclude"]:
                r = torch.arange(len(d2), device=DEV)
                d2[r, r + i] = math.inf
            out[i:i + step] = d2.topk(case["k"], dim=1, largest=False).values
        return None, out.sqrt()
    if kind in ("rays", "occlusion"):
        if float(case["n"]) * case["tris"] > 8e9:
            return None
        v, t, o, d = _ray_inputs(case, seed)
        limit = math.inf if kind == "rays" else case["reach"]
        time, nrm = _rays64(v, t, o, d, limit)
        hit = torch.isfinite(time)
        if kind == "occlusion":
            return hit.to(torch.uint8)
        return None, torch.where(hit, time, torch.full_like(time, -1.0)), nrm
    if kind == "sample":
        v, t = _ellipsoids(case["ellipsoids"], _gen(seed, 7))
        pos, nrm = _sample64(v, t, case["n"], seed & 0xFFFF)
        return pos, nrm, None
    if kind == "batch":
        verts, tris, queries = _batch_inputs(case, seed)
        if sum(float(len(t)) * len(q) for t, q in zip(tris, queries)) > 4e9:
            return None
        return None, torch.cat([_closest64(v, t, q, -1.0)[0] for v, t, q in zip(verts, tris, queries)])
    if kind == "icp":
        src, target = _icp_inputs(case, seed)
        if float(case["n"]) * case["target"] * case["starts"] * case["iterations"] > 1e11:
            return None
        tr, err = _icp64(src, target, _rotations(case["starts"]), case["iterations"])
        return tr, err, None
    return None  # served requests: mixed outputs of the kinds above
