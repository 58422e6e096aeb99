"""GPU tests of thg_icp_align (Thea's Icp3::align) against the numpy restatement in oracle/icp.py
with the oracle's kd-tree as the nearest-point search: same iteration counts, transforms within
1e-9, errors within 1e-9 relative; a batch of K starting transforms gives each problem exactly the
result of aligning it alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _ellipsoid(g, n, axes=(1.0, 0.6, 0.3)):
    u = g.normal(size=(n, 3))
    return (u / np.linalg.norm(u, axis=1)[:, None] * np.array(axes)).astype(np.float32)


def _axis_rot(axis, angle):
    ax = np.asarray(axis, np.float64) / np.linalg.norm(axis)
    K = np.array([[0, -ax[2], ax[1]], [ax[2], 0, -ax[0]], [-ax[1], ax[0], 0]])
    return np.eye(3) + np.sin(angle) * K + (1 - np.cos(angle)) * K @ K


def _xf(R, t):
    return np.hstack([R, np.asarray(t, np.float64).reshape(3, 1)])


def _check(tr, err, its, ref, label):
    rtr, rerr, rits = ref
    assert its == rits, f"{label}: iterations {its} vs {rits}"
    assert np.allclose(tr, rtr, rtol=0, atol=1e-9), f"{label}: transform differs by {np.abs(tr - rtr).max()}"
    assert abs(err - rerr) <= 1e-9 * max(abs(rerr), 1e-30), f"{label}: error {err} vs {rerr}"


@pytest.mark.parametrize("kabsch", [False, True])
def test_icp_points_matches_oracle(oracle, kabsch):
    import thea_amd
    from oracle import icp as I
    print(f"case icp points kabsch={kabsch}", flush=True)
    g = np.random.default_rng(11)
    to = _ellipsoid(g, 30000)
    src = to[::7].astype(np.float64) @ _axis_rot([1, 2, 3], 0.08).T + np.array([0.02, -0.01, 0.03])
    bvh = thea_amd.PointBvh(to)
    icp = thea_amd.Icp3(kabsch=kabsch)
    tr, err, its = icp.alignBatch(src, bvh)
    kd = oracle.KdTree(points=to)
    ref = I.icp_align(lambda x: kd.closest(x, mode=0)[1], src, kabsch=kabsch)
    _check(tr[0], err[0], its[0], ref, "points")
    if kabsch:
        assert err[0] < 0.2 * I.measure_error(I.identity(), src, kd.closest(src.astype(np.float32), mode=0)[1])


def test_icp_batch_equals_single_and_oracle(oracle):
    import thea_amd
    from oracle import icp as I
    print("case icp batch", flush=True)
    g = np.random.default_rng(12)
    to = _ellipsoid(g, 20000)
    src = to[::5].astype(np.float64) + 0.01
    inits = np.stack([_xf(_axis_rot(g.normal(size=3), a), g.normal(size=3) * 0.05)
                      for a in (0.0, 0.05, 0.3, 1.0, 2.5, 3.1)])
    bvh = thea_amd.PointBvh(to)
    icp = thea_amd.Icp3(kabsch=True)
    tr, err, its = icp.alignBatch(src, bvh, initial=inits)
    kd = oracle.KdTree(points=to)
    for k in range(len(inits)):
        t1, e1, i1 = icp.alignBatch(src, bvh, initial=inits[k:k + 1])
        assert np.array_equal(t1[0], tr[k]) and e1[0] == err[k] and i1[0] == its[k], f"problem {k}"
        ref = I.icp_align(lambda x: kd.closest(x, mode=0)[1], I.xf_apply(inits[k], src), kabsch=True)
        _check(tr[k], err[k], its[k], ref, f"problem {k}")


@pytest.mark.parametrize("target", ["points", "mesh"])
def test_icp_problems_that_end_apart_equal_single(target):
    """200,000 positions while all four problems run, which are searched in spatial order, and 100,000 or
    fewer once two have ended, which are searched as they come."""
    import thea_amd
    from thea_amd import workloads as W
    print(f"case icp ending apart {target}", flush=True)
    g = np.random.default_rng(15)
    n = 50000
    if target == "points":
        to = _ellipsoid(g, n)
        src = to.astype(np.float64)
        bvh = thea_amd.PointBvh(to)
    else:
        v, t = W.torus(96, 48, R=1.0, r=0.3, amp=0.03, seed=7)
        src = (v[t[g.integers(0, len(t), n)]] * g.dirichlet([1, 1, 1], n)[:, :, None]).sum(1)
        bvh = thea_amd.MeshBvh(thea_amd.Mesh(v, t))
    inits = np.stack([_xf(_axis_rot([1, 2, 3], a), [d, -d, 0.5 * d])
                      for a, d in ((0.01, 0.002), (0.1, 0.02), (0.3, 0.05), (0.9, 0.1))])
    icp = thea_amd.Icp3(fractional_error_threshold=0.05, max_iterations=25, kabsch=True)
    tr, err, its = icp.alignBatch(src, bvh, initial=inits)
    its = list(its)
    assert sorted(its)[1] < sorted(its)[3], its  # two or fewer problems search on
    for k in range(len(inits)):
        t1, e1, i1 = icp.alignBatch(src, bvh, initial=inits[k:k + 1])
        assert i1[0] == its[k] and e1[0] == err[k] and np.array_equal(t1[0], tr[k]), f"problem {k}"


def test_icp_more_coordinates_than_one_launch_holds():
    """63 of 64 problems search on with 23,000,000 points each: 1.45e9 correspondences, whose coordinates
    are more than the 2^32 threads of one launch (118 GB)."""
    import torch
    import thea_amd
    if torch.cuda.mem_get_info()[0] < 150 << 30:
        pytest.skip("needs 150 GB of device memory")
    print("case icp 63 x 23,000,000", flush=True)
    g = np.random.default_rng(17)
    to = _ellipsoid(g, 40)
    src = to[np.arange(23_000_000) % len(to)].astype(np.float64)
    move = _xf(_axis_rot([1, 2, 3], 0.9), [0.1, -0.1, 0.05])
    inits = np.stack([_xf(np.eye(3), [0, 0, 0])] + 63 * [move])
    bvh = thea_amd.PointBvh(to)
    icp = thea_amd.Icp3(min_iterations=2, max_iterations=2, kabsch=True)
    tr, err, its = icp.alignBatch(src, bvh, initial=inits)
    t1, e1, i1 = icp.alignBatch(src, bvh, initial=inits[1:2])
    torch.cuda.synchronize()
    bvh.ctx.trim()
    assert its[0] == 0 and i1[0] == 2 and np.all(its[1:] == 2)
    assert np.all(err[1:] == e1[0]) and np.all(tr[1:] == t1[0])


def test_icp_leaves_other_streams_running():
    """Whatever its arrays take (340 MB here), an alignment waits for its own stream only."""
    import time
    import torch
    import thea_amd
    print("case icp beside another stream", flush=True)
    g = np.random.default_rng(16)
    src = _ellipsoid(g, 500_000).astype(np.float64)
    bvh = thea_amd.PointBvh(_ellipsoid(g, 1000))
    inits = np.repeat(_xf(np.eye(3), [0, 0, 0])[None], 10, 0)
    icp = thea_amd.Icp3(min_iterations=1, max_iterations=1, kabsch=True)
    icp.alignBatch(src, bvh, initial=inits)  # memory and code in place
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    torch.cuda._sleep(10_000_000)
    torch.cuda.synchronize()
    cycles = int(10_000_000 / (time.perf_counter() - t0))  # in one second, roughly
    for _ in range(8):
        s = torch.cuda.Stream()
        done = torch.cuda.Event()
        with torch.cuda.stream(s):
            torch.cuda._sleep(cycles)
            done.record()
        bvh.closestPoint(np.zeros((1, 3), np.float32))
        if done.query():  # shares a hardware queue with the default stream
            continue
        icp.alignBatch(src, bvh, initial=inits)
        beside = not done.query()
        torch.cuda.synchronize()
        assert beside
        return
    pytest.skip("no stream runs beside the default stream")


def test_icp_mesh_weights_up(oracle):
    import thea_amd
    from oracle import icp as I
    from thea_amd import workloads as W
    print("case icp mesh", flush=True)
    v, t = W.torus(96, 48, R=1.0, r=0.3, amp=0.03, seed=7)
    g = np.random.default_rng(13)
    sampler = thea_amd.MeshSampler(thea_amd.Mesh(v, t))
    pts, _, _ = sampler.sampleEvenlyByArea(8000, seed=3)
    src = pts.astype(np.float64) @ _axis_rot([0, 0, 1], 0.1).T + np.array([0.05, 0.0, 0.0])
    wt, wr = g.uniform(0.5, 1.5, len(src)), g.uniform(0.5, 1.5, len(src))
    bvh = thea_amd.MeshBvh(thea_amd.Mesh(v, t))
    icp = thea_amd.Icp3(max_iterations=15, kabsch=True)
    icp.setUpVector([0, 0, 2.0])
    tr, err, its = icp.alignBatch(src, bvh, translation_weights=wt, rotation_weights=wr)
    kd = oracle.KdTree(v, t)
    ref = I.icp_align(lambda x: kd.closest(x, mode=0)[1], src, max_it=15, wt=wt, wr=wr, up=[0, 0, 1.0], kabsch=True)
    _check(tr[0], err[0], its[0], ref, "mesh")
    assert np.allclose(tr[0][2, :3], [0, 0, 1], atol=1e-12)


def test_icp_edge_cases():
    import thea_amd
    from thea_amd import _capi as capi
    print("case icp edge cases", flush=True)
    g = np.random.default_rng(14)
    to = _ellipsoid(g, 1000)
    bvh = thea_amd.PointBvh(to)
    icp = thea_amd.Icp3()
    tr, err = icp.align(np.zeros((0, 3)), bvh)
    assert np.array_equal(tr, np.hstack([np.eye(3), np.zeros((3, 1))])) and err == 0
    tr, err, its = icp.alignBatch(to.astype(np.float64), bvh)
    assert its[0] == 0 and err[0] == 0 and np.array_equal(tr[0], np.hstack([np.eye(3), np.zeros((3, 1))]))
    empty = thea_amd.PointBvh(np.zeros((0, 3), np.float32))
    with pytest.raises(capi.TheaGpuError) as e:
        icp.align(to.astype(np.float64), empty)
    assert e.value.code == capi.THG_E_INVALID
