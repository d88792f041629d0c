"""Labels of pixels far from every site: few points in wide empty textures, every size class of the
far kernels, against brute force with ties to the lower column, then the lower row."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _check(ctx, xy, T, step):
    labels, pix, nf = ctx.voronoi(xy, T)
    px, py = (pix >> 16).astype(np.int32), (pix & 0xffff).astype(np.int32)
    sites = np.unique(labels)
    sites = sites[np.lexsort((py[sites], px[sites]))]
    Y = np.arange(T, dtype=np.int32)[None, :]
    for x0 in range(0, T, 64 * step):   # every step-th band of 64 columns
        X = np.arange(x0, min(x0 + 64, T), dtype=np.int32)[:, None]
        best = np.full((len(X), T), 1 << 30, dtype=np.int32)
        who = np.zeros((len(X), T), dtype=np.int64)
        for s in sites:
            d = (X - px[s]) ** 2 + (Y - py[s]) ** 2
            np.copyto(who, s, where=d < best)
            np.minimum(best, d, out=best)
        assert np.array_equal(who, labels[x0:x0 + 64])


@pytest.mark.parametrize("T,step", [(64, 1), (128, 1), (256, 1), (512, 1), (1024, 3), (2048, 5), (4096, 9), (8192, 17)])
def test_sparse_texture(T, step):
    import galpha2d_amd as G
    ctx = G.Context(0)
    rng = np.random.default_rng(T)
    corners = np.array([[0.0, 0.0], [1.0, 1.0]])
    spots = {"few": rng.random((5, 2)), "corner": 0.03 * rng.random((40, 2)), "column": np.c_[np.full(30, 0.5), rng.random(30)],
             "row": np.c_[rng.random(30), np.full(30, 0.25)], "grid": np.stack(np.meshgrid(*[np.arange(1, 5) / 5] * 2), -1).reshape(-1, 2)}
    for name, p in spots.items():
        print("case:", T, name, flush=True)
        _check(ctx, np.concatenate([corners, p]), T, step)
    ctx.close()
