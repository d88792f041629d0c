"""Alpha results on the host: gathered together up to 16 MiB, array by array above, of a single run and of
the sets of a batch (unaligned parts of the arrays); they stay valid after later calls."""
import gc

import numpy as np
import pytest

from galpha2d_amd import datagen

pytestmark = pytest.mark.gpu


def _same(a, b):
    assert a.keys() <= b.keys()   # (the oracle reports more)
    for k in a:
        assert a[k].dtype == b[k].dtype and np.array_equal(a[k], b[k]), k


@pytest.mark.parametrize("n", [0, 1, 3, 5, 1000, 40003, 70001])
def test_host_call(oracle, n):
    import galpha2d_amd as G
    print("case: host call", n, flush=True)
    xy = datagen.uniform(n + 1, n)
    T = G.auto_texture(n)
    tris, alpha = G.compute_alpha_shapes(xy, T)
    kept = {k: v.copy() for k, v in alpha.items()}
    G.compute_alpha_shapes(datagen.uniform(9, 2000), 512)   # overwrites the staging and the device arrays
    gc.collect()
    _same(alpha, kept)
    assert np.array_equal(tris, oracle.delaunay(xy)[0])
    _same(alpha, oracle.alpha(xy, tris))
    if n:
        alpha["vert_nu_min"][0] = 7   # writable


def test_batch_sets():
    import galpha2d_amd as G
    sets = [datagen.uniform(k, 301 + 37 * k) for k in range(5)]
    ctx = G.Context(0)
    tris = ctx.batch(sets, with_alpha=True)
    for k, xy in enumerate(sets):
        print("case: set", k, flush=True)
        t, a = G.compute_alpha_shapes(xy, G.auto_texture(len(xy)))
        assert np.array_equal(t, tris[k])
        _same(ctx.batch_alpha(k), a)
    ctx.close()
