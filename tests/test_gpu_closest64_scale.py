"""The double search's float reject test at coordinates where float arithmetic underflows, overflows or
carries a large offset: answers must stay those of the double brute force, bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scale", [1e-30, 1e-20, 1.0, 1e15, 1e19, 1e25])
@pytest.mark.parametrize("offset", [0.0, 1e3, 1e7])
@pytest.mark.parametrize("leaf", [1, 16])
def test_scales_and_offsets(oracle, scale, offset, leaf):
    import thea_amd
    g = np.random.default_rng(7)
    pts = (g.normal(size=(3_000, 3)) + offset) * scale
    pts[50:60] = pts[:10]
    q = (g.normal(size=(2_001, 3)) * 1.5 + offset) * scale
    q[:100] = pts[:100]
    b = thea_amd.PointBvhF64(pts, leaf_size=leaf)
    for bound in (-1.0, 0.3 * scale, 0.0):
        idx, _, _, d2 = b.closest(q, dist_bound=bound, want_d2=True)
        ridx, rd2 = oracle.brute_closest_points_f64(pts, q, bound)
        assert np.array_equal(idx, ridx), (scale, offset, bound)
        assert np.array_equal(d2[ridx >= 0], rd2[ridx >= 0])
