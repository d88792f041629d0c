"""Frame removal on shapes whose vertices nearly all lie on one arc or line: every box of boundary vertices touches the
circles and lines of the search, and the exact predicates decide.  Against the oracle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _arc(n, part, seed):
    a = np.random.default_rng(seed).random(n) * 2 * np.pi * part
    return np.stack([np.cos(a), np.sin(a)], 1)


def _sides(n, slope):
    t = np.random.default_rng(n).permutation(n // 2) / 65536.0
    a = np.stack([t, slope * t], 1)
    return np.concatenate([a, a + [0, 1 / 1024]])


def _near_line(n, seed):
    t = np.random.default_rng(seed).random(n)
    return np.stack([t, 0.3 * t], 1)


CASES = {
    "half circle 3,000": lambda: (_arc(3000, 0.5, 1), 256),
    "half circle 12,000": lambda: (_arc(12000, 0.5, 2), 512),
    "quarter circle 5,000": lambda: (_arc(5000, 0.25, 3), 512),
    "half circle and its centre": lambda: (np.concatenate([_arc(3000, 0.5, 4), [[0.0, 0.0], [0.0, -0.5]]]), 512),
    "axis-parallel sides": lambda: (_sides(20000, 0.0), 1024),
    "sloped sides": lambda: (_sides(20000, 0.375), 1024),
    "line and two points": lambda: (np.concatenate([_sides(6000, 0.375)[:3000], [[0.3, 0.7], [0.1, -1.0]]]), 256),
    "near a line": lambda: (_near_line(2000, 5), 256),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_shapes(oracle, name):
    import galpha2d_amd as G
    print("case:", name, flush=True)
    xy, T = CASES[name]()
    ctx = G.Context(0)
    got, ref = ctx.delaunay(xy, T), oracle.delaunay(xy)[0]
    assert got.shape == ref.shape and np.array_equal(got, ref)
    ctx.close()


def test_batch(oracle):
    import galpha2d_amd as G
    print("case: batch of shapes", flush=True)
    sets = [CASES[k]()[0][:6000] for k in sorted(CASES)]
    ctx = G.Context(0)
    for xy, tris in zip(sets, ctx.batch(sets)):
        assert np.array_equal(tris, oracle.delaunay(xy)[0])
    ctx.close()
