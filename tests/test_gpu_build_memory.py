"""Block reuse between builds and the box pyramid at its level edges.

A freed device block serves the next allocation of about its size; meshes built one after another in
growing, shrinking and repeated sizes, with queries of the previous mesh still queued when it is
freed, must give the results of a fresh build, also from several threads.
"""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(n, seed):
    g = np.random.default_rng(seed)
    c = g.random((n, 1, 3), dtype=np.float32)
    v = (c + g.random((n, 3, 3), dtype=np.float32) * np.float32(0.02)).reshape(-1, 3)
    return v, np.arange(3 * n, dtype=np.int32).reshape(-1, 3)


@pytest.mark.parametrize("n", [1, 2, 255, 256, 257, 511, 65_535, 65_536, 65_537, 131_071, 131_073])
@pytest.mark.parametrize("leaf", [1, 8])
def test_boxes_at_level_edges(n, leaf):
    import thea_amd
    g = np.random.default_rng(n)
    p = g.normal(size=(n, 3)).astype(np.float32)
    b = thea_amd.PointBvh(p, leaf_size=leaf)
    f, i, ids = b.export()
    lo, hi = f[:, [0, 1, 2, 6, 7, 8]].reshape(-1, 2, 3), f[:, [3, 4, 5, 9, 10, 11]].reshape(-1, 2, 3)
    ref, cnt = i[:, 12:14], i[:, 14:16]
    sp = p[ids]
    assert np.array_equal(np.sort(ids), np.arange(n))
    for c in range(2):
        for k in np.flatnonzero((ref[:, c] < 0) & (cnt[:, c] > 0)):
            e = sp[~ref[k, c]: ~ref[k, c] + cnt[k, c]]
            assert np.array_equal(lo[k, c], e.min(0)) and np.array_equal(hi[k, c], e.max(0))
        inner = np.flatnonzero(ref[:, c] >= 0)
        assert np.array_equal(lo[inner, c], lo[ref[inner, c]].min(1))
        assert np.array_equal(hi[inner, c], hi[ref[inner, c]].max(1))


def _rounds(sizes, out, ctx):
    import torch
    import thea_amd
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        for k, n in enumerate(sizes):
            v, t = _mesh(n, k)
            q = torch.from_numpy(np.random.default_rng(k).random((20_000, 3), dtype=np.float32)).cuda()
            b = thea_amd.MeshBvh(thea_amd.Mesh(v, t, ctx=ctx))
            out.append(b.closestPoint(q))
            del b  # its queries may still be running
        s.synchronize()


def test_reused_blocks_give_fresh_results():
    import thea_amd
    sizes = [40_000, 36_000, 44_000, 40_000, 33_000, 90_000, 40_000]
    ctx = thea_amd.default_context()
    outs = [[] for _ in range(3)]
    threads = [threading.Thread(target=_rounds, args=(sizes, o, ctx)) for o in outs]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    for k, n in enumerate(sizes):
        v, t = _mesh(n, k)
        q = np.random.default_rng(k).random((20_000, 3), dtype=np.float32)
        want = thea_amd.MeshBvh(thea_amd.Mesh(v, t)).closestPoint(q)
        for o in outs:
            for a, b in zip(o[k], want):
                assert np.array_equal(a.cpu().numpy(), b), (k, n)


def test_blocks_are_given_back_with_a_context():
    import torch
    import thea_amd
    ctx = thea_amd.Context(0)
    free0 = torch.cuda.mem_get_info()[0]
    v, t = _mesh(300_000, 1)
    for _ in range(2):
        m = thea_amd.Mesh(v, t, ctx=ctx)
        b = thea_amd.MeshBvh(m)
        b.close()
        m.close()
    ctx.close()
    # what is left: the stream-ordered pool's share of the build's temporaries (256 MB at most)
    assert free0 - torch.cuda.mem_get_info()[0] <= 300 << 20


def test_trim_gives_back_kept_memory():
    """The default context, which lives as long as the process, gives back what it keeps on request."""
    import torch
    import thea_amd
    ctx = thea_amd.default_context()
    v, t = _mesh(300_000, 1)

    def build():
        m = thea_amd.Mesh(v, t)
        b = thea_amd.MeshBvh(m)
        r = b.closestPoint(v[:1000])
        b.close()
        m.close()
        return r

    want = build()
    ctx.trim()
    free0 = torch.cuda.mem_get_info()[0]
    build()
    held = free0 - torch.cuda.mem_get_info()[0]
    ctx.trim()
    left = free0 - torch.cuda.mem_get_info()[0]
    print(f"held {held >> 20} MB, after trim {left >> 20} MB", flush=True)
    assert held >= 64 << 20  # the arrays over elements alone are 72 MB
    assert left <= 8 << 20
    for a, b in zip(build(), want):
        assert np.array_equal(a, b)
