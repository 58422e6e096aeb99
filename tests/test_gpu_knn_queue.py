"""The work-queue k-NN kernel (and closest points of point BVHs) against the wave walk and the oracle.

A batch of more than max(4 queries per triangle, 2^18) on a mesh, or max(1 per 2 points, 2^17) on
points and any of more than 2^19 there, takes the wave walk up to k = 16; smaller ones, down to lower lines on trees of fewer than
8,000 elements, and every k above 16, take the queue. Both must give the canonical lists. Sizes are the edges of its waves (1 to 32 queries each, by k), k the
edges of its list widths, and trees of fewer elements than k leave slots empty.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _equal(a, b, label):
    for x, y in zip(a, b):
        assert np.array_equal(np.asarray(x).view(np.uint32), np.asarray(y).view(np.uint32)), label


@pytest.fixture(scope="module")
def mesh_case():
    import thea_amd
    from thea_amd import workloads as W
    v, t = W.torus(90, 45)  # 8,100 triangles: the queue up to 2^18
    g = np.random.default_rng(11)
    lo, hi = W.inflated_box(v, 1.2)
    q = g.uniform(lo, hi, size=((1 << 18) + 1, 3)).astype(np.float32)
    q[3] = np.nan
    return thea_amd.MeshBvh(thea_amd.Mesh(v, t)), q


@pytest.mark.parametrize("k", [1, 2, 5, 8, 9, 16])
def test_mesh_lists_equal_wave_walk(mesh_case, k):
    b, q = mesh_case
    ref = b.kClosestElements(q, k, want_d2=True)
    refb = b.kClosestElements(q, k, dist_bound=0.15, want_d2=True)
    for n in (1, 7, 33, 4_097, 12_801, 51_201, 131_073, (1 << 18) - 1, 1 << 18):
        _equal(b.kClosestElements(q[:n], k, want_d2=True), [x[:n] for x in ref], f"k={k} n={n}")
    _equal(b.kClosestElements(q[:900], k, dist_bound=0.15, want_d2=True), [x[:900] for x in refb], f"k={k} bound")


@pytest.mark.parametrize("k", [1, 4, 16, 17, 32])
@pytest.mark.parametrize("n", [1, 130, 9_000])
def test_mesh_lists_equal_oracle(oracle, k, n):
    import thea_amd
    from thea_amd import workloads as W
    v, t = W.geodesic_sphere(3)
    v, t = np.concatenate([v, v * np.float32(0.5)]), np.concatenate([t, t + len(v), t[:50]])  # 50 duplicates
    g = np.random.default_rng(n)
    q = g.uniform(-1.5, 1.5, size=(n, 3)).astype(np.float32)
    idx, _, d2 = thea_amd.MeshBvh(thea_amd.Mesh(v, t), leaf_size=2).kClosestElements(q, k, want_d2=True)
    m = min(n, 400)
    ridx, rd2, _ = oracle.KdTree(v, t).knn(q[:m], k, mode=0)
    _equal((idx[:m], d2[:m]), (ridx, rd2), f"k={k} n={n}")


@pytest.mark.parametrize("count", [1, 2, 3, 5, 31, 70])
@pytest.mark.parametrize("exclude", [False, True])
def test_small_point_sets(oracle, count, exclude):
    import thea_amd
    g = np.random.default_rng(count)
    p = g.normal(size=(count, 3)).astype(np.float32)
    p[count // 2] = p[0]  # an exact duplicate
    b = thea_amd.PointBvh(p, leaf_size=2)
    d2all = ((p[:, None] - p[None]) ** 2)
    d2all = d2all[..., 0] + (d2all[..., 1] + d2all[..., 2])
    for k in (1, 3, 8, 32):
        idx, _, d2 = b.kClosestElements(p, k, exclude_self=exclude, want_d2=True)
        for i in range(count):
            order = sorted((d2all[i, j], j) for j in range(count) if not (exclude and j == i))[:k]
            want = [j for _, j in order] + [-1] * (k - len(order))
            assert idx[i].tolist() == want, (count, k, i)
            assert np.array_equal(d2[i][:len(order)], np.array([d for d, _ in order], np.float32))


@pytest.mark.parametrize("leaf", [1, 4, 16])
def test_points_equal_wave_walk(leaf):
    import thea_amd
    g = np.random.default_rng(leaf)
    p = g.normal(size=(30_000, 3)).astype(np.float32)
    p[20_000:20_100] = p[:100]
    b = thea_amd.PointBvh(p, leaf_size=leaf)
    q = (g.normal(size=((1 << 17) + 1, 3)) * 1.2).astype(np.float32)
    q[:500] = p[:500]
    q[9] = np.inf
    ref = b.closest(q, want_d2=True)
    refk = b.kClosestElements(q, 6, want_d2=True)
    for n in (1, 40, 4_097, 1 << 17):
        _equal(b.closest(q[:n], want_d2=True), [x[:n] for x in ref], f"closest n={n}")
        _equal(b.kClosestElements(q[:n], 6, want_d2=True), [x[:n] for x in refk], f"k-NN n={n}")
    assert (b.closest(q[:50], dist_bound=0.0)[0] == -1).all()


@pytest.mark.parametrize("k", [1, 6])
def test_large_point_sets_at_the_line(k):
    """2^19 queries of 1,100,000 points take the queue, one more the wave walk."""
    import torch
    import thea_amd
    g = torch.Generator(device="cuda").manual_seed(k)
    p = torch.randn(1_100_000, 3, generator=g, device="cuda")
    b = thea_amd.PointBvh(p)
    q = torch.randn((1 << 19) + 1, 3, generator=g, device="cuda") * 1.3
    q[:1000] = p[:1000]
    for x, y in zip(b.kClosestElements(q, k, want_d2=True), b.kClosestElements(q[:-1], k, want_d2=True)):
        assert torch.equal(x[:-1], y)
    if k == 1:
        for x, y in zip(b.closestPoint(q), b.closestPoint(q[:-1])):
            assert torch.equal(x[:-1], y)


def test_more_threads_than_one_launch_holds():
    """From 2^29 queries on, the 8 threads that a query of a list of more than 16 takes add up to more
    than the 2^32 of one launch (51 GB here: 6 of queries, 37 of indices, 9 to sort them)."""
    import torch
    import thea_amd
    from thea_amd import _capi as capi
    n, k = (1 << 29) + 1_001, 17
    if torch.cuda.mem_get_info()[0] < 80 << 30:
        pytest.skip("needs 80 GB of device memory")
    b = thea_amd.PointBvh(np.random.default_rng(1).random((40, 3), dtype=np.float32))
    g = torch.Generator(device="cuda").manual_seed(1)
    q = torch.rand(n, 3, generator=g, device="cuda")
    idx = torch.full((n, k), -2, dtype=torch.int32, device="cuda")
    print(f"case n={n} k={k}", flush=True)
    stream = torch.cuda.current_stream().cuda_stream
    capi.check(capi.lib().thg_k_closest(b.h, q.data_ptr(), n, k, -1.0, 0, idx.data_ptr(), None, None,
                                        capi.THG_MEM_DEVICE, stream))
    for a in range(0, n, 1 << 27):
        assert bool((idx[a:a + (1 << 27)] >= 0).all()), a
    for a in (0, (1 << 28) - 500, (1 << 29) - 500, n - 1_000):
        assert torch.equal(idx[a:a + 1_000], b.kClosestElements(q[a:a + 1_000].contiguous(), k)[0]), a
    del q, idx
    torch.cuda.empty_cache()
    b.ctx.trim()
