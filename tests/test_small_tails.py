"""Small sets that the single-workgroup stages hand over to grid launches: many vertices left to move or delete (points on a
spiral), and long flip lists of points that nearly all share pixels.  Triangles against the oracle, and
the launches that say who did the work."""
import numpy as np
import pytest

from galpha2d_amd import datagen

pytestmark = pytest.mark.gpu


def _spiral(n, seed):
    t = np.sqrt(np.random.default_rng(seed).random(n)) * 40
    return np.stack([t * np.cos(t), t * np.sin(t)], 1)


def _one_pixel(n, seed):
    p = np.random.default_rng(seed).random((n, 2)) * 1e-9
    p[:2] = [[1.0, 1.0], [-1.0, 0.5]]
    return p


CASES = [("spiral 2,000", "k_shift_greedy", lambda: _spiral(2000, 1), True),
         ("spiral 8,000", "k_shift_greedy", lambda: _spiral(8000, 2), True),
         ("spiral 1,000", "k_shift_greedy", lambda: _spiral(1000, 3), False),
         ("uniform 8,000", "k_shift_greedy", lambda: datagen.uniform(4, 8000), False),
         ("one pixel 2,000", "k_flip_test", lambda: _one_pixel(2000, 5), True),
         ("one pixel 300", "k_flip_test", lambda: _one_pixel(300, 6), False),
         ("uniform 2,000", "k_flip_test", lambda: datagen.uniform(7, 2000), False)]


@pytest.mark.parametrize("name,kernel,make,grid", CASES, ids=[c[0] for c in CASES])
def test_small(oracle, name, kernel, make, grid):
    import galpha2d_amd as G
    print("case:", name, flush=True)
    xy = make()
    ctx = G.Context(0)
    out = []
    probe = ctx.kernel_probe(kernel, lambda: out.append(ctx.delaunay(xy, G.auto_texture(len(xy)))))
    assert np.array_equal(out[0], oracle.delaunay(xy)[0])
    assert (probe["launches"] > 0) == grid
    ctx.close()
