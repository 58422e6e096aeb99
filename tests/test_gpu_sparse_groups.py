"""GPU parity of the work queue's sparse batches, in which a wave takes 64 >> lg queries.

One 500k-triangle closed surface at leaf size 1 (about 500k leaves) with queries uniform in its
inflated box, so most queries lie inside it, far from the nearest triangle, and meet a large part of
the tree. Dense batches (more than 786,432 closest-point queries, more than 4 k-NN queries per
triangle, more than 131,072 queries of 120,000 points or more) take one walk per wave; subsets of the
same queries of 100 ... 100,000 take the queue at each width. Bar: every row of every subset
bit-identical to the dense result (indices, squared distances, closest points), and the dense result
and the smallest subset bit-identical to the oracle.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# subset sizes: 1 (up to 6,400), 2, 4, 8, 16 queries per wave for closest points; k-NN lists of up to 16
# spread twice as far: 1 (up to 12,800), 2, 4, 8
SUBSETS = [100, 3000, 6000, 12000, 24000, 50000, 100_000]
DENSE = 800_000


@pytest.fixture(scope="module")
def sphere():
    import thea_amd
    from thea_amd import workloads as W
    g = np.random.default_rng(41)
    v, t = W.uv_sphere(354, 708)
    v = (v * (1 + 0.02 * g.normal(size=len(v)))[:, None]).astype(np.float32)
    t = t.astype(np.int32)
    lo, hi = W.inflated_box(v, 1.2)
    q = g.uniform(lo, hi, size=(4 * len(t) + 1, 3)).astype(np.float32)
    b = thea_amd.MeshBvh(thea_amd.Mesh(v, t), leaf_size=1)
    perm = g.permutation(DENSE)
    print(f"case sphere: {len(t)} tris, bvh {b.info}", flush=True)
    assert DENSE > max(1.25 * len(t), 786_432), "sizes no longer select the intended kernels"
    return v, t, q, b, perm


def _same(a, b_, label):
    assert np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b_).view(np.uint32)), label


def test_closest_subsets_equal_dense(sphere, oracle):
    v, t, q, b, perm = sphere
    idx, dist, cp, d2 = b.closest(q[:DENSE], want_d2=True)
    for n in SUBSETS:
        sel = perm[:n]
        print(f"case closest subset n={n}", flush=True)
        i2, dist2, cp2, d22 = b.closest(q[sel], want_d2=True)
        assert np.array_equal(i2, idx[sel]), f"n={n}: {np.count_nonzero(i2 != idx[sel])} index mismatches"
        _same(d22, d2[sel], f"n={n}: d2")
        _same(cp2, cp[sel], f"n={n}: closest points")
        _same(dist2, dist[sel], f"n={n}: dist")
    sel = perm[:100]
    kd = oracle.KdTree(v, t)
    ridx, rcp, rd2, _ = kd.closest(q[sel], mode=0)
    assert np.array_equal(idx[sel], ridx)
    _same(d2[sel], rd2, "oracle d2")
    _same(cp[sel], rcp, "oracle closest points")


def test_closest_subsets_with_bound(sphere):
    v, t, q, b, perm = sphere
    bound = 0.05  # most queries inside the sphere find nothing within it
    idx, _, cp, d2 = b.closest(q[:DENSE], dist_bound=bound, want_d2=True)
    assert 0 < np.count_nonzero(idx >= 0) < DENSE
    for n in (100, 6000, 50000):
        sel = perm[:n]
        print(f"case closest bound subset n={n}", flush=True)
        i2, _, cp2, d22 = b.closest(q[sel], dist_bound=bound, want_d2=True)
        assert np.array_equal(i2, idx[sel])
        hit = i2 >= 0
        _same(d22[hit], d2[sel][hit], f"n={n}: d2")
        _same(cp2[hit], cp[sel][hit], f"n={n}: cp")


@pytest.mark.parametrize("k", [3, 8, 16])
def test_knn_subsets_equal_dense(sphere, oracle, k):
    v, t, q, b, perm = sphere
    idx, dist, d2 = b.kClosestElements(q, k, want_d2=True)
    for n in SUBSETS:
        sel = perm[:n]
        print(f"case knn k={k} subset n={n}", flush=True)
        i2, dist2, d22 = b.kClosestElements(q[sel], k, want_d2=True)
        assert np.array_equal(i2, idx[sel]), f"n={n}: {np.count_nonzero(i2 != idx[sel])} index mismatches"
        _same(d22, d2[sel], f"n={n}: d2")
        _same(dist2, dist[sel], f"n={n}: dist")
    sel = perm[:100]
    ridx, rd2, _ = oracle.KdTree(v, t).knn(q[sel], k, mode=0)
    assert np.array_equal(idx[sel], ridx)
    _same(d2[sel], rd2, "oracle d2")


def test_points_subsets_equal_dense(sphere, oracle):
    import thea_amd
    v, _, _, _, _ = sphere
    g = np.random.default_rng(43)
    pts = v[g.permutation(len(v))[:240_000]]
    pts = np.concatenate([pts, pts[:500]])  # exact duplicates: ties on equal distance
    pb = thea_amd.PointBvh(pts, leaf_size=1)
    lo, hi = pts.min(0) * 1.2, pts.max(0) * 1.2
    q = g.uniform(lo, hi, size=(140_000, 3)).astype(np.float32)
    q[:300] = pts[:300]
    assert len(q) > max(len(pts) / 2, 1 << 17)
    idx, _, cp, d2 = pb.closest(q, want_d2=True)
    kidx, _, kd2 = pb.kClosestElements(q, 6, want_d2=True)
    for n in (100, 3000, 6000, 100_000):
        sel = np.arange(n)
        print(f"case points subset n={n}", flush=True)
        i2, _, cp2, d22 = pb.closest(q[sel], want_d2=True)
        assert np.array_equal(i2, idx[sel])
        _same(d22, d2[sel], "points d2")
        _same(cp2, cp[sel], "points cp")
        k2, _, kd22 = pb.kClosestElements(q[sel], 6, want_d2=True)
        assert np.array_equal(k2, kidx[sel])
        _same(kd22, kd2[sel], "points knn d2")
    ridx, rd2, _ = oracle.KdTree(points=pts).knn(q[:100], 6, mode=0)
    assert np.array_equal(kidx[:100], ridx)
    _same(kd2[:100], rd2, "oracle points knn d2")
