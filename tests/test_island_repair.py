"""Repair of the discrete Voronoi diagram around sites that fail the island certificate: labels against
brute force with phase 3's ties (lower column, then lower row), the certificate itself, and
triangulations of batches where only some sets are repaired."""
import numpy as np
import pytest

from galpha2d_amd import datagen

pytestmark = pytest.mark.gpu


def _clusters(n, seed):
    return datagen.gaussian_clusters(np.random.default_rng(seed), n, 4, 0.01)


def _check_labels(ctx, T, n):
    repaired = 0
    X, Y = np.meshgrid(np.arange(T), np.arange(T), indexing="ij")
    for seed in range(8):
        print("case: clusters", T, n, seed, flush=True)
        labels, pix, nf = ctx.voronoi(_clusters(n, seed), T)
        repaired += ctx.stats()["islandSites"]
        px, py = (pix >> 16).astype(np.int64), (pix & 0xffff).astype(np.int64)
        sites = np.unique(labels)
        best = np.full((T, T), 1 << 60, dtype=np.int64)
        who = np.zeros((T, T), dtype=np.int64)
        for s in sites[np.lexsort((py[sites], px[sites]))]:   # lower column, then lower row first
            d = (X - px[s]) ** 2 + (Y - py[s]) ** 2
            np.copyto(who, s, where=d < best)
            np.minimum(best, d, out=best)
        assert np.array_equal(who, labels)
        # certificate: the same label one step toward the site
        dx, dy = np.sign(px[labels] - X), np.sign(py[labels] - Y)
        ok = (dx == 0) & (dy == 0)
        for ux, uy in ((dx, 0), (0, dy), (dx, dy)):
            ux, uy = np.broadcast_to(ux, X.shape), np.broadcast_to(uy, X.shape)
            ok |= ((ux != 0) | (uy != 0)) & (labels[X + ux, Y + uy] == labels)
        assert ok.all()
    return repaired


def test_labels():
    """The sizes together must hold repaired sites (the smallest textures may have none)."""
    import galpha2d_amd as G
    ctx = G.Context(0)
    assert sum(_check_labels(ctx, T, n) for T, n in ((64, 500), (128, 900), (256, 2500), (1024, 300))) > 0
    ctx.close()


@pytest.mark.parametrize("nsets", [1, 7, 33])
def test_batches(oracle, nsets):
    import galpha2d_amd as G
    print("case: batch of", nsets, flush=True)
    sets = [_clusters(300 + 211 * k, k) if k % 3 != 1 else datagen.uniform(k, 500 + 97 * k) for k in range(nsets)]
    ctx = G.Context(0)
    for xy, tris in zip(sets, ctx.batch(sets)):
        assert np.array_equal(tris, oracle.delaunay(xy)[0])
    assert ctx.stats()["islandSites"] > 0
    ctx.close()
