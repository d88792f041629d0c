"""Canonical order where runs of equal 32-bit keys are long (one vertex with thousands of neighbours numbered close
together, among more than 2^20 points): the order is made with whole keys, and only there."""
import numpy as np
import pytest

from galpha2d_amd import datagen

pytestmark = pytest.mark.gpu


def _hub(n, spokes, seed, at=0):
    """Point `at` with `spokes` neighbours numbered next to it, the other points away from it."""
    rng = np.random.default_rng(seed)
    ang = rng.permutation(spokes) * (2 * np.pi / spokes) + rng.uniform(0, 1e-6, spokes)
    rest = rng.uniform(-1, 1, (2 * n, 2))
    rest = rest[np.hypot(rest[:, 0], rest[:, 1]) > 0.3][:n - spokes - 1]
    return np.concatenate([rest[:at], [[0.0, 0.0]], 0.25 * np.c_[np.cos(ang), np.sin(ang)], rest[at:]])


def _check(tris, hub, spokes):
    t, v = tris[:, :3], tris[:, 3:6].astype(np.int64)
    assert (v[:, 0] < v[:, 1:].min(axis=1)).all()
    assert (np.diff((v[:, 0] << 32) | v[:, 1]) > 0).all()
    assert int((v[:, 0] == hub).sum()) >= spokes - 1
    back = np.arange(len(t))
    for i in range(3):
        has = t[:, i] >= 0
        assert (t[t[has, i] >> 2, t[has, i] & 3] >> 2 == back[has]).all()


@pytest.mark.parametrize("n,spokes,at,whole", [(1100000, 20000, 0, 1), (1100000, 20000, 700000, 1), (1100000, 300, 0, 0),
                                               (300000, 20000, 0, 0), (1100000, 0, 0, 0)])
def test_runs(n, spokes, at, whole):
    import galpha2d_amd as G
    print("case: hub", n, spokes, at, flush=True)
    ctx = G.Context(0)
    xy = _hub(n, spokes, n, at) if spokes else datagen.uniform(3, n)
    d = G.DeviceBuffer(np.ascontiguousarray(xy))
    probe = ctx.kernel_probe("k_canon_keys", lambda: ctx.compute_device(d.ptr, n, G.auto_texture(n)))
    assert probe["launches"] == whole
    if spokes:
        _check(ctx.triangles(), at, spokes)
        assert ctx.stats()["nTris"] == len(ctx.triangles())
    d.free()
    ctx.close()


def test_batch():
    import galpha2d_amd as G
    print("case: hubs of a batch", flush=True)
    ctx = G.Context(0)
    sizes = ((700000, 9000, 0), (5000, 300, 10), (400000, 5000, 1000))
    sets = [_hub(n, s, n, at) for n, s, at in sizes]
    for xy, tris, (n, spokes, at) in zip(sets, ctx.batch(sets), sizes):
        _check(tris, at, spokes)
        assert np.array_equal(tris, ctx.delaunay(xy, G.auto_texture(n)))
    ctx.close()
