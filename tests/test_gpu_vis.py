"""GPU tests of thg_visibility (Visibility::compute) against the oracle: the same rays, the same
hits, the same fractions."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("num_rays,explicit_scale", [(100, False), (37, True)])
def test_visibility_matches_oracle(oracle, num_rays, explicit_scale):
    import thea_amd
    from thea_amd import workloads as W
    print(f"case visibility rays={num_rays} scale={explicit_scale}", flush=True)
    v, t = W.torus(192, 96, R=1.0, r=0.3, amp=0.05, seed=4)
    mesh = thea_amd.Mesh(v, t)
    pos, _, _ = thea_amd.MeshSampler(mesh).sampleEvenlyByArea(5000, seed=5)
    b = thea_amd.MeshBvh(mesh)
    lo, hi = b.getBounds()
    e = hi - lo
    default_scale = np.float32(np.sqrt(e[0] * e[0] + (e[1] * e[1] + e[2] * e[2])))
    scale = 2.5 if explicit_scale else None
    vis = b.visibility(pos, num_rays=num_rays, seed=11, scale=scale)
    ref = oracle.visibility(oracle.KdTree(v, t), pos, num_rays, default_scale if scale is None else scale, 11)
    assert np.array_equal(vis, ref)
    # a surface point of a closed mesh sees at most half the sphere
    assert vis.max() <= 0.75 and 0.2 < vis.mean() < 0.55


def test_visibility_device_and_chunks(oracle):
    import torch
    import thea_amd
    from thea_amd import workloads as W
    print("case visibility device", flush=True)
    v, t = W.torus(64, 32, seed=1)
    mesh = thea_amd.Mesh(v, t)
    pos, _, _ = thea_amd.MeshSampler(mesh).sampleEvenlyByArea(2000, seed=2)
    b = thea_amd.MeshBvh(mesh)
    host = b.visibility(pos, num_rays=64, seed=3)
    dev = b.visibility(torch.as_tensor(pos, device="cuda"), num_rays=64, seed=3)
    assert dev.is_cuda and np.array_equal(dev.cpu().numpy(), host)
    # 1,700 points x 10,000 rays: more than one 2^24-ray chunk
    many = b.visibility(pos[:1700], num_rays=10000, seed=4, scale=2.0)
    assert np.array_equal(many, oracle.visibility(oracle.KdTree(v, t), pos[:1700], 10000, 2.0, 4))
    assert len(b.visibility(np.zeros((0, 3), np.float32))) == 0


def test_one_ray_per_lane_sorts_its_rays(oracle):
    """Where the work queue is not used (THG_RAY_Q4=0, read once per process), the rays are put in order,
    one sort per chunk, and the fractions stay the same."""
    import os
    import subprocess
    import sys
    import thea_amd
    from thea_amd import workloads as W
    print("case visibility one ray per lane", flush=True)
    code = ("import sys, numpy as np, thea_amd; from thea_amd import workloads as W;"
            "v, t = W.torus(64, 32, seed=1); b = thea_amd.MeshBvh(thea_amd.Mesh(v, t)); b.ctx.set_timing(True);"
            "x = b.visibility(v[:500], num_rays=64, seed=3);"
            "print(b.ctx.kernel_time('order')[1], b.ctx.kernel_time('any_hit')[1], x.tobytes().hex())")
    out = subprocess.run([sys.executable, "-c", code], env=dict(os.environ, THG_RAY_Q4="0"), capture_output=True,
                         text=True, timeout=120, check=True,
                         cwd=os.path.dirname(os.path.dirname(os.path.abspath(__file__)))).stdout.split()
    assert out[0] == "1" and out[1] == "1"
    v, t = W.torus(64, 32, seed=1)
    b = thea_amd.MeshBvh(thea_amd.Mesh(v, t))
    assert bytes.fromhex(out[2]) == b.visibility(v[:500], num_rays=64, seed=3).tobytes()
