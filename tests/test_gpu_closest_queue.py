"""The work-queue closest-triangle kernel against the compacted wave walk and the oracle.

Batches of up to 1.25 queries per triangle take the queue, and on small meshes up to 65,536 + 64 per
triangle (at least 131,072, at most 786,432); larger ones take the wave walk, and both must give the
canonical bits. Sizes are the edges of its waves (1 to 32 queries per wave)
and of its rule; the equidistant sphere makes every query at its centre meet the whole tree, so the
stack runs into its throttle.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WAVE_N = 786_433  # takes the wave walk on every mesh of fewer than 629,146 triangles


def _equal(a, b, label):
    for x, y in zip(a, b):
        assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32)), label


@pytest.fixture(scope="module", params=[1, 4, 16])
def torus(request):
    import thea_amd
    from thea_amd import workloads as W
    v, t = W.torus(128, 64)  # 16,384 triangles: the queue up to WAVE_N - 1
    b = thea_amd.MeshBvh(thea_amd.Mesh(v, t), leaf_size=request.param)
    g = np.random.default_rng(7)
    lo, hi = W.inflated_box(v, 1.2)
    q = g.uniform(lo, hi, size=(WAVE_N, 3)).astype(np.float32)
    q[5] = np.nan
    q[11, 1] = np.inf
    return b, q, b.closest(q, want_d2=True), b.closest(q, dist_bound=0.1, want_d2=True)


@pytest.mark.parametrize("n", [1, 2, 31, 32, 33, 64, 4_095, 4_097, 6_400, 6_401, 12_801, 51_201, 102_401, 131_072, 131_073, 204_801, 262_143, 262_144,
                               524_287, 524_288, WAVE_N - 1])
def test_queue_equals_wave_walk(torus, n):
    b, q, ref, ref_bound = torus
    _equal(b.closest(q[:n], want_d2=True), [x[:n] for x in ref], f"n={n}")
    _equal(b.closest(q[:n], dist_bound=0.1, want_d2=True), [x[:n] for x in ref_bound], f"n={n} bound")


def test_zero_bound_and_tiny_meshes():
    import thea_amd
    v = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, 0, 1]], np.float32)
    t = np.array([[0, 1, 2], [0, 2, 3], [0, 3, 1]], np.int32)
    q = np.random.default_rng(3).normal(size=(100, 3)).astype(np.float32)
    for leaf in (1, 4):
        b = thea_amd.MeshBvh(thea_amd.Mesh(v, t), leaf_size=leaf)
        assert (b.closest(q, dist_bound=0.0)[0] == -1).all()
        big = np.tile(q, (7_900, 1))
        i0, d0, c0, _ = b.closest(q)
        i1, d1, c1, _ = b.closest(big)
        _equal((i0, d0, c0), (i1[:100], d1[:100], c1[:100]), f"leaf {leaf}")


@pytest.mark.parametrize("n", [1, 40, 5_000])
def test_equidistant_queries_fill_the_stack(oracle, n):
    import thea_amd
    from thea_amd import workloads as W
    v, t = W.uv_sphere(150, 300)
    v = v.astype(np.float32)
    b = thea_amd.MeshBvh(thea_amd.Mesh(v, t), leaf_size=1)
    q = (np.random.default_rng(n).normal(size=(n, 3)) * 1e-5).astype(np.float32)
    idx, _, cp, d2 = b.closest(q, want_d2=True)
    m = min(n, 200)
    ridx, rcp, rd2, _ = oracle.KdTree(v, t).closest(q[:m], mode=0)
    _equal((idx[:m], cp[:m], d2[:m]), (ridx, rcp, rd2), f"n={n}")


def test_plan_with_both_kernels():
    import torch
    import thea_amd
    from thea_amd import batch
    from thea_amd import workloads as W
    g = np.random.default_rng(9)
    meshes, queries = [], []
    for tris, n in ((300, 50), (2_000, WAVE_N), (8_000, 3_000), (2, 33), (50_000, 70_000)):
        v, t = W._mesh_of_size(tris, len(meshes) % 2, g) if tris > 2 else \
            (np.eye(3, dtype=np.float32), np.array([[0, 1, 2], [0, 2, 1]], np.int32))
        lo, hi = W.inflated_box(v, 1.2)
        meshes.append((v, t))
        queries.append(g.uniform(lo, hi, size=(n, 3)).astype(np.float32))
    nv, nt, nq, verts, tris, qs = batch.concat(meshes, queries)
    plan = batch.BatchPlan(nv, nt, nq)
    dv, dt, dq = (torch.from_numpy(x).cuda() for x in (verts, tris, qs))
    for _ in range(3):
        idx, dist = plan.run(dv, dt, dq)
        off = 0
        for (v, t), q in zip(meshes, queries):
            i, d, _ = thea_amd.MeshBvh(thea_amd.Mesh(v, t)).closestPoint(q)
            _equal((idx[off:off + len(q)].cpu().numpy(), dist[off:off + len(q)].cpu().numpy()), (i, d), f"{len(q)}")
            off += len(q)
