"""The work-queue ray kernels against the oracle and against themselves in other batches.

A batch of n rays is spread over waves of 8 to 64 rays (8 up to 32,768 rays, 16 up to 65,536, 32 up to
131,072, then 64), so the sizes are one wave, its edges and the edges of that rule. A ray's answer must not
depend on the wave it runs in: rays parallel to an axis, NaN rays and rays that start on the surface
(hits at time 0) share waves with ordinary ones.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [1, 7, 8, 9, 63, 64, 65, 32_768, 32_769, 65_537, 131_072]


def _bits(x):
    x = np.asarray(x)
    return x.view(np.uint32) if x.dtype == np.float32 else x


def _equal(a, b, label):
    for x, y in zip(a, b):
        assert np.array_equal(_bits(x), _bits(y)), label


def _rays(v, t, n, seed):
    g = np.random.default_rng(seed)
    lo, hi = v.min(0) - 0.2, v.max(0) + 0.2
    o = g.uniform(lo, hi, size=(n, 3)).astype(np.float32)
    d = g.normal(size=(n, 3)).astype(np.float32)
    d[::5] = np.eye(3, dtype=np.float32)[g.integers(0, 3, len(d[::5]))]  # parallel to an axis
    o[::7] = v[t[g.integers(0, len(t), len(o[::7]))]].mean(1)             # from the surface
    o[::11] = v[g.integers(0, len(v), len(o[::11]))]                      # from its vertices
    d[13::1000] = np.nan
    o[17::1000] = np.inf
    d[19::1000] = 0
    return o, d


@pytest.mark.parametrize("leaf", [1, 4, 16])
def test_answers_do_not_depend_on_the_wave(oracle, leaf):
    import thea_amd
    from thea_amd import workloads as W
    v, t = W.torus(40, 20)
    b = thea_amd.MeshBvh(thea_amd.Mesh(v, t), leaf_size=leaf)
    o, d = _rays(v, t, SIZES[-1] + 1, leaf)
    for mt in (-1.0, 0.7, 0.0):
        ref = b.rayStructureIntersection(o, d, mt)
        hit = b.rayIntersects(o, d, mt)
        assert np.array_equal(hit.astype(bool), ref[0] >= 0), mt
        for n in SIZES:
            s = SIZES[-1] + 1 - n
            _equal(b.rayStructureIntersection(o[s:], d[s:], mt), [x[s:] for x in ref], f"first n={n} max={mt}")
            _equal([b.rayIntersects(o[s:], d[s:], mt)], [hit[s:]], f"any n={n} max={mt}")
    kd = oracle.KdTree(v, t)
    idx, tm, nrm = b.rayStructureIntersection(o[:3_000], d[:3_000])
    ok = np.isfinite(o[:3_000]).all(1) & np.isfinite(d[:3_000]).all(1) & (d[:3_000] != 0).any(1)
    ridx, rt = kd.ray(o[:3_000][ok], d[:3_000][ok])[:2]
    _equal((idx[ok], tm[ok]), (ridx, rt), "oracle")


@pytest.mark.parametrize("count", [1, 2, 3, 5])
def test_smallest_trees(oracle, count):
    import thea_amd
    v = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [1, 1, 0.1]], np.float32)
    t = np.array([[0, 1, 2], [1, 3, 2], [0, 1, 2], [0, 3, 2], [2, 1, 0]], np.int32)[:count]  # duplicates
    b = thea_amd.MeshBvh(thea_amd.Mesh(v, t), leaf_size=1)
    o, d = _rays(v, t, 200, count)
    ok = np.isfinite(o).all(1) & np.isfinite(d).all(1) & (d != 0).any(1)
    o, d = o[ok], d[ok]
    idx, tm, _ = b.rayStructureIntersection(o, d)
    _equal((idx, tm), oracle.KdTree(v, t).ray(o, d)[:2], count)
    assert np.array_equal(b.rayIntersects(o, d).astype(bool), idx >= 0)


def test_shared_centroids_make_a_deep_tree(oracle):
    """Clusters at doubling distances: a walk of many levels, each of which leaves entries on the stack."""
    import thea_amd
    g = np.random.default_rng(2)
    p = (2.0 ** -np.arange(28))[:, None, None] * (1 + 0.3 * g.random((28, 40, 3)))
    tri = (p.reshape(-1, 1, 3) + 0.02 * p.reshape(-1, 1, 3) * g.normal(size=(p.shape[0] * 40, 3, 3))).astype(np.float32)
    v, t = tri.reshape(-1, 3), np.arange(tri.shape[0] * 3, dtype=np.int32).reshape(-1, 3)
    b = thea_amd.MeshBvh(thea_amd.Mesh(v, t), leaf_size=1)
    n = 4_097
    o = (g.random((n, 3)) * 1.5).astype(np.float32)
    d = (tri[g.integers(0, len(tri), n)].mean(1) - o).astype(np.float32)
    idx, tm, _ = b.rayStructureIntersection(o, d)
    _equal((idx, tm), oracle.KdTree(v, t).ray(o, d)[:2], "deep")
    assert np.array_equal(b.rayIntersects(o, d).astype(bool), idx >= 0)


def test_sorted_batch_equals_its_halves():
    """More than 2^22 rays on a tree of more than 256 MB are traced in spatial order."""
    import torch
    import thea_amd
    from thea_amd import workloads as W
    v, t = W.torus(2400, 1200)  # 5,760,000 triangles of 48 bytes
    dev = "cuda"
    b = thea_amd.MeshBvh(thea_amd.Mesh(torch.as_tensor(v, device=dev), torch.as_tensor(t, device=dev)), leaf_size=4)
    g = torch.Generator(device=dev).manual_seed(3)
    n = (1 << 22) + 1
    o = (torch.rand(n, 3, generator=g, device=dev) * 2 - 1) * float(np.abs(v).max())
    d = torch.randn(n, 3, generator=g, device=dev)
    whole = b.rayStructureIntersection(o, d) + (b.rayIntersects(o, d),)
    for s in (slice(0, n // 2), slice(n // 2, n)):
        o1, d1 = o[s].contiguous(), d[s].contiguous()
        half = b.rayStructureIntersection(o1, d1) + (b.rayIntersects(o1, d1),)
        for x, y in zip(whole, half):
            assert torch.equal(x[s], y)
