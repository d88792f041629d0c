"""Canonical order with 32-bit sort keys: triangles of one vertex whose second vertices have close
input indices share a key, up to a thousand here, and are still in (v0, v1) order, each with links
that lead back."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _hub(n, spokes, seed):
    """Point 0 with `spokes` neighbours numbered next to it, the other points away from it."""
    rng = np.random.default_rng(seed)
    ang = rng.permutation(spokes) * (2 * np.pi / spokes) + rng.uniform(0, 1e-4, spokes)
    rest = rng.uniform(-1, 1, (n, 2))
    rest = rest[np.hypot(rest[:, 0], rest[:, 1]) > 0.3][:n - spokes - 1]
    return np.concatenate([[[0.0, 0.0]], 0.25 * np.c_[np.cos(ang), np.sin(ang)], rest])


def _check(tris, spokes):
    t, v = tris[:, :3], tris[:, 3:6].astype(np.int64)
    assert (v[:, 0] < v[:, 1:].min(axis=1)).all()
    key = (v[:, 0] << 32) | v[:, 1]
    assert (np.diff(key) > 0).all()
    assert int((v[:, 0] == 0).sum()) >= spokes
    back = np.arange(len(t))
    for i in range(3):
        has = t[:, i] >= 0
        u, j = t[has, i] >> 2, t[has, i] & 3
        assert (t[u, j] >> 2 == back[has]).all()


@pytest.mark.parametrize("n,spokes", [(70000, 500), (300000, 900), (1100000, 1000)])
def test_hub(n, spokes):
    import galpha2d_amd as G
    print("case: hub", n, spokes, flush=True)
    ctx = G.Context(0)
    _check(ctx.delaunay(_hub(n, spokes, n)), spokes)
    ctx.close()


def test_hub_batch():
    import galpha2d_amd as G
    print("case: hubs of a batch", flush=True)
    ctx = G.Context(0)
    for tris, spokes in zip(ctx.batch([_hub(n, s, n) for n, s in ((700000, 800), (5000, 300), (400000, 700))]), (800, 300, 700)):
        _check(tris, spokes)
    ctx.close()
