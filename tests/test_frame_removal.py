"""Frame removal (gift wrapping over the boundary vertices) against the oracle, on boundaries
where it has to do the most: long straight sides with points just outside, every point on the hull,
regions that fall apart without the frame, and boundary vertex counts on both sides of one box (64) and of
one step of boxes (4,096)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _straight_sides(n, out, seed):
    """Points on the sides of a square (collinear runs), a few inside, and `out` points just outside:
    the pockets between a straight side and a hull edge to an outside point are long and thin."""
    rng = np.random.default_rng(seed)
    t = rng.permutation(8192)[:n] / 8192.0
    k = n // 4
    sides = [np.stack([t[:k], np.zeros(k)], 1), np.stack([np.ones(k), t[k:2 * k]], 1),
             np.stack([t[2 * k:3 * k], np.ones(k)], 1), np.stack([np.zeros(n - 3 * k), t[3 * k:]], 1)]
    far = np.stack([rng.random(out), -0.001 - 0.001 * rng.random(out)], 1)
    return np.concatenate(sides + [rng.random((n // 8, 2)), far])


def _circle(n, seed):
    a = np.random.default_rng(seed).random(n) * 2 * np.pi
    return np.stack([np.cos(a), np.sin(a)], 1)


def _islands(groups, per, seed):
    """Tight groups far apart (the real triangles of different groups touch only frame triangles)."""
    rng = np.random.default_rng(seed)
    return (rng.random((groups, 1, 2)) + 1e-4 * rng.random((groups, per, 2))).reshape(-1, 2)


CASES = {
    "sides 12": lambda: (_straight_sides(12, 1, 1), 64),
    "sides 900": lambda: (_straight_sides(900, 2, 2), 512),
    "sides 1500": lambda: (_straight_sides(1500, 1, 3), 512),
    "sides 6000": lambda: (_straight_sides(6000, 5, 4), 1024),
    "circle 1000": lambda: (_circle(1000, 5), 512),
    "circle 60": lambda: (_circle(60, 6), 256),
    "circle 70": lambda: (_circle(70, 6), 256),
    "circle 5000": lambda: (_circle(5000, 7), 1024),
    "far from the origin": lambda: (_circle(3000, 12) * 1e-3 + [1e6, -1e6], 1024),
    "lone points": lambda: (_islands(40, 1, 8), 2048),
    "pairs": lambda: (_islands(30, 2, 9), 256),
    "two points and a far group": lambda: (np.concatenate([_islands(1, 50, 10), [[9.0, 9.0], [9.0, -7.0]]]), 256),
    "collinear": lambda: (np.array([[k * 0.25, 0.5 + k * 0.125] for k in range(60)]), 256),
    "collinear and one": lambda: (np.array([[k * 0.25, 0.5 + k * 0.125] for k in range(60)] + [[7.0, 1.0]]), 256),
    "grid": lambda: (np.array([(i / 40.0, j / 40.0) for i in range(41) for j in range(41)]), 512),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_boundaries(oracle, name):
    import galpha2d_amd as G
    print("case:", name, flush=True)
    xy, T = CASES[name]()
    ctx = G.Context(0)
    ref, _ = oracle.delaunay(xy)
    got = ctx.delaunay(xy, T)
    assert got.shape == ref.shape and np.array_equal(got, ref)
    ctx.close()


@pytest.mark.parametrize("big", [False, True])
def test_batch(oracle, big):
    """All of them, or the small ones, as one batch."""
    import galpha2d_amd as G
    print("case: batch", big, flush=True)
    sets = [CASES[k]()[0] for k in sorted(CASES) if big or CASES[k]()[0].shape[0] < 1000]
    ctx = G.Context(0)
    for xy, tris in zip(sets, ctx.batch(sets)):
        ref, _ = oracle.delaunay(xy)
        assert np.array_equal(tris, ref.reshape(-1, 9))
    ctx.close()
