"""Shifting, deletion and insertion of small and larger sets (one workgroup up to 8,192 points, launches
above) on coarse textures, where many vertices cannot move or share a pixel, against the oracle."""
import numpy as np
import pytest

from galpha2d_amd import datagen

pytestmark = pytest.mark.gpu


def _points(kind, n):
    rng = np.random.default_rng(n)
    if kind == "uniform":
        return datagen.uniform(n, n)
    if kind == "clusters":
        return datagen.gaussian_clusters(rng, n, 5, 0.004)
    if kind == "star":      # a hub with many neighbours in every pixel round it, and a far ring
        a = rng.uniform(0, 2 * np.pi, n)
        r = np.where(rng.random(n) < 0.7, 1e-3, 1.0) * (1 + 1e-3 * rng.random(n))
        return np.concatenate([[[0.0, 0.0]], np.c_[r * np.cos(a), r * np.sin(a)]])[:n]
    side = int(np.ceil(np.sqrt(n)))   # a lattice turned by a little: thin triangles, exact ties broken by rounding
    i, j = np.meshgrid(np.arange(side), np.arange(side))
    p = np.c_[i.ravel(), j.ravel()][:n].astype(float)
    return p @ np.array([[np.cos(0.3), -np.sin(0.3)], [np.sin(0.3), np.cos(0.3)]])


@pytest.mark.parametrize("kind", ["uniform", "clusters", "star", "lattice"])
@pytest.mark.parametrize("n,T", [(3, 64), (40, 64), (700, 64), (2048, 64), (2049, 128), (8192, 128), (8193, 128), (20000, 256)])
def test_coarse_texture(oracle, kind, n, T):
    import galpha2d_amd as G
    print("case: shifting", kind, n, T, flush=True)
    ctx = G.Context(0)
    xy = _points(kind, n)
    for _ in range(2):   # the second run on the buffers and tags that the first left
        assert np.array_equal(ctx.delaunay(xy, T), oracle.delaunay(xy)[0])
    ctx.close()
