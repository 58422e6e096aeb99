"""The radix sort behind the tree build and the query order, at the sizes where its tiles change.

Build: a point BVH's leaf order is the stable order of the points' 30-bit Morton codes, so it must
equal numpy's stable argsort of codes computed with the same float operations. Queries: a batch and
its reverse visit different orders of the same queries, so every query's answer must be the same
bits either way (an order that lost or repeated a query would leave one unanswered). Float batches are
sorted above 131,072 queries, double ones from 4,096 on; ray batches only above 2^22 on trees of more
than 256 MB (test_gpu_ray_queue.py).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [2, 63, 255, 257, 1_023, 1_024, 1_025, 4_097, 65_537, (1 << 20) - 1, 1 << 20, (1 << 20) + 1, 2_100_003]


def _spread(v):
    v = v & 0x3FF
    for s, m in ((16, 0x030000FF), (8, 0x0300F00F), (4, 0x030C30C3), (2, 0x09249249)):
        v = (v | (v << s)) & m
    return v


def _morton(p):
    lo, hi = p.min(0), p.max(0)
    inv = np.where(hi - lo > 0, np.float32(1) / np.where(hi - lo > 0, hi - lo, 1).astype(np.float32), 0).astype(np.float32)
    c = np.clip((p - lo) * inv * np.float32(1024), 0, 1023).astype(np.uint32)
    return (_spread(c[:, 0]) << 2) | (_spread(c[:, 1]) << 1) | _spread(c[:, 2])


@pytest.mark.parametrize("n", SIZES)
def test_build_order_is_the_stable_morton_order(n):
    import thea_amd
    rng = np.random.default_rng(n)
    p = rng.random((n, 3), dtype=np.float32)
    p[rng.integers(0, n, n // 3)] = p[0]  # equal codes must keep input order
    _, _, ids = thea_amd.PointBvh(p, leaf_size=1).export()
    assert np.array_equal(ids, np.argsort(_morton(p), kind="stable").astype(np.int32))


@pytest.mark.parametrize("n", [131_073, 200_001, (1 << 18) - 1, 1 << 18, 786_433, 1 << 20, (1 << 20) + 1, 2_500_001])
def test_query_order_answers_every_query(n):
    import torch
    import thea_amd
    from thea_amd import workloads as W
    v, t = W.torus(64, 32)
    bvh = thea_amd.MeshBvh(thea_amd.Mesh(v, t))
    g = torch.Generator(device="cuda").manual_seed(n)
    q = (torch.rand(n, 3, generator=g, device="cuda") - 0.5) * 3.5
    i0, d0 = bvh.closestElementWithDistance(q)
    i1, d1 = bvh.closestElementWithDistance(q.flip(0))
    assert torch.equal(i0, i1.flip(0)) and torch.equal(d0, d1.flip(0))


@pytest.mark.parametrize("n", [4_096, 4_097, 65_537, 100_001, (1 << 20) + 1])
def test_double_query_order_answers_every_query(n):
    import thea_amd
    g = np.random.default_rng(n)
    bvh = thea_amd.PointBvhF64(g.normal(size=(5_000, 3)))
    q = g.normal(size=(n, 3))
    for a, b in zip(bvh.closest(q)[:3], bvh.closest(q[::-1])[:3]):
        assert np.array_equal(a, b[::-1])
