"""Frame removal where nearly every point lies on the boundary of what the frame triangles cover: more demands
than unused triangle slots, on flat curves, whose triangles are found from two and three sides at once."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _curve(n, height, seed=6):
    t = np.random.default_rng(seed).random(n) * 20
    return np.stack([t, height * np.sin(t)], 1)


@pytest.mark.parametrize("n,height", [(20000, 0.1), (40000, 0.1), (20000, 0.03)])
def test_flat_curve(oracle, n, height):
    import galpha2d_amd as G
    print("case: flat curve", n, height, flush=True)
    xy = _curve(n, height)
    ctx = G.Context(0)
    assert np.array_equal(ctx.delaunay(xy, 1024), oracle.delaunay(xy)[0])
    ctx.close()


def test_batch(oracle):
    import galpha2d_amd as G
    print("case: flat curves of a batch", flush=True)
    sets = [_curve(n, h, n) for n, h in ((9000, 0.1), (700, 0.2), (12000, 0.05), (10000, 0.1), (64, 0.1), (11000, 0.15))]
    ctx = G.Context(0)
    for xy, tris in zip(sets, ctx.batch(sets)):
        assert np.array_equal(tris, oracle.delaunay(xy)[0])
    ctx.close()
