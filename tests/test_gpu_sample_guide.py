"""Area sampling through the guide table against the oracle, where its ranges hold no, one or very
many triangles: triangle counts around its size steps, runs of zero-area triangles, one triangle with
nearly all the area, and areas that grow by powers of two (which also leave the exact-scan path)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(areas, seed):
    g = np.random.default_rng(seed)
    n = len(areas)
    o = g.random((n, 1, 3)).astype(np.float32)
    e = np.zeros((n, 3, 3), np.float32)
    e[:, 1, 0] = np.sqrt(2 * np.asarray(areas))
    e[:, 2, 1] = np.sqrt(2 * np.asarray(areas))
    return (o + e).reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.int32).reshape(-1, 3)


def _areas(kind, n):
    g = np.random.default_rng(n)
    if kind == "even":
        return np.full(n, 0.01)
    if kind == "zeros":
        a = g.random(n) * 0.01
        a[n // 4: n // 2] = 0.0
        a[0] = a[-1] = 0.0
        a[n // 3 if n < 3 else 1] = 0.5
        return a
    if kind == "one":
        a = np.full(n, 1e-9)
        a[n // 2] = 10.0
        return a
    return 2.0 ** -(np.arange(n) % 60)


@pytest.mark.parametrize("kind", ["even", "zeros", "one", "powers"])
@pytest.mark.parametrize("n", [1, 2, 3, 255, 256, 257, 1_024, 1_025, 70_000])
def test_samples_equal_oracle(oracle, kind, n):
    import thea_amd
    v, t = _mesh(_areas(kind, n), 3)
    got = thea_amd.MeshSampler(thea_amd.Mesh(v, t)).sampleEvenlyByArea(60_000, seed=9, stream_id=2)
    want = oracle.sample_area(v, t, 60_000, 9, 2)
    assert len(got[0]) == len(want[0])
    for a, b in zip(got, want):
        assert np.array_equal(np.asarray(a).view(np.uint32), np.asarray(b).view(np.uint32))
