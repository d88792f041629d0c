"""A repair of the discrete diagram takes no memory that a context without one has not taken."""
import ctypes

import numpy as np
import pytest

from galpha2d_amd import datagen

pytestmark = pytest.mark.gpu


def _free(G):
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert G.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0   # (of the library's own HIP runtime)
    return free.value


def test_memory():
    """Arrays of a texture take 67 MB here (4 bytes per pixel)."""
    import galpha2d_amd as G
    print("case: memory of a repair", flush=True)
    ctx = G.Context(0)
    grid = np.stack(np.meshgrid(np.arange(141.0), np.arange(141.0)), -1).reshape(-1, 2)
    ctx.delaunay(grid, 4096)
    assert ctx.stats()["islandSites"] == 0
    free = _free(G)
    for seed in range(20):
        ctx.delaunay(datagen.gaussian_clusters(np.random.default_rng(seed), len(grid), 4, 0.01), 4096)
        if ctx.stats()["islandSites"] > 0:
            break
    assert ctx.stats()["islandSites"] > 0
    assert free - _free(G) < 48 << 20
    ctx.close()
