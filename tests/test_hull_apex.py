"""The apex search of frame removal (hull_apex of mesh.hip) on the host: its text, one wave of 64 lanes
as 64 fibers in lock step, must find the same apex for a set and for the set scaled by a power of two (the
exact predicates are free of scale), and the apex that rational arithmetic finds."""
import os
import subprocess
from fractions import Fraction

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "galpha2d_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"
HARNESS = r"""
#include <hip/hip_runtime.h>
#include <ucontext.h>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <functional>
#include <vector>
#include "dev_common.h"
#include "kernels.h"
// a wave: every lane is a fiber, and every collective ends with all lanes having given their value
static int g_lane;
static ucontext_t g_main, g_ctx[64];
static unsigned long long g_val[2][64];
static int g_phase[64];
static long long g_steps;   // of all lanes
static void meet() { g_steps++; swapcontext(&g_ctx[g_lane], &g_main); }
template <class T> static T exchange(T v, int from)
{
    const int l = g_lane, p = g_phase[l]++ & 1;
    unsigned long long w = 0;
    memcpy(&w, &v, sizeof(T));
    g_val[p][l] = w;
    meet();
    T r;
    memcpy(&r, &g_val[p][from & 63], sizeof(T));
    return r;
}
static unsigned long long h_ballot(bool b)
{
    const int l = g_lane, p = g_phase[l]++ & 1;
    g_val[p][l] = b;
    meet();
    unsigned long long m = 0;
    for (int k = 0; k < 64; k++) m |= g_val[p][k] << k;
    return m;
}
#define __ballot(x) h_ballot(x)
#define __any(x) (h_ballot(x) != 0)
#define __shfl(v, k, w) exchange(v, k)
#define __shfl_xor(v, k, w) exchange(v, g_lane ^ (k))
#define atomicOr(p, v) (*(p) |= (v))
#define __ffsll(x) __builtin_ffsll(x)
#define __popcll(x) __builtin_popcountll(x)
typedef unsigned long long u64;
static int orient_dev(const MeshDev &m, double2 a, double2 b, double2 c)
{
    int ovf = 0;
    const int s = orient_sign(a, b, c, &ovf);
    if (ovf) *m.status = 1;
    return s;
}
static inline int incircle_at(const MeshDev &m, double2 a, double2 b, double2 c, double2 d, int ia, int ib, int ic, int id)
{
    const int s = incircle_filter(a, b, c, d);
    if (s) return s;
    int ovf = 0;
    const int t = incircle_exact_sos(a, ia, b, ib, c, ic, d, id, &ovf);
    if (ovf) *m.status = 1;
    return t;
}
#undef GA_INLINE
#define GA_INLINE static inline
#undef __device__
#define __device__
#undef __noinline__
#define __noinline__
#include "hull.h"
static std::function<void(int)> g_body;
static void fiber() { g_body(g_lane); g_phase[g_lane] = -1; swapcontext(&g_ctx[g_lane], &g_main); }
static void wave(std::function<void(int)> body)
{
    static std::vector<char> stacks(64 * 65536);
    g_body = body;
    for (int l = 0; l < 64; l++) {
        getcontext(&g_ctx[l]);
        g_ctx[l].uc_stack.ss_sp = &stacks[65536 * l];
        g_ctx[l].uc_stack.ss_size = 65536;
        g_ctx[l].uc_link = nullptr;
        makecontext(&g_ctx[l], fiber, 0);
        g_phase[l] = 0;
    }
    for (bool more = true; more;) {
        more = false;
        for (g_lane = 0; g_lane < 64; g_lane++)
            if (g_phase[g_lane] >= 0) {
                swapcontext(&g_main, &g_ctx[g_lane]);
                more = more || g_phase[g_lane] >= 0;
            }
    }
}
// argv[1]: n, demands, the set's snap scale, the vertices of another set before it, n points, demands (p, q); prints the apexes, then
// the nearest vertices of the demands' first ends, the status and the number of collectives
int main(int, char **argv)
{
    FILE *f = fopen(argv[1], "r");
    int n, nd, other, status = 0;
    SetDesc sd{};
    if (fscanf(f, "%d %d %la %d", &n, &nd, &sd.scale, &other) != 4) return 1;
    std::vector<double2> pos(n + 1);
    std::vector<int> ids(n + 1), zero(n + 1);
    std::vector<HullBox> box(n / 64 + 1, HullBox{INFINITY, INFINITY, -INFINITY, -INFINITY});
    for (int i = 0; i < n; i++) {
        if (fscanf(f, "%la %la", &pos[i].x, &pos[i].y) != 2) return 1;
        ids[i] = i;
        HullBox &b = box[i / 64];
        b.lx = fmin(b.lx, pos[i].x); b.hx = fmax(b.hx, pos[i].x);
        b.ly = fmin(b.ly, pos[i].y); b.hy = fmax(b.hy, pos[i].y);
    }
    ids[n] = n;
    sd.poff = other;
    sd.n = n - other;
    MeshDev m{};
    m.n = n; m.pos = pos.data(); m.status = &status; m.sets = &sd; m.vset = zero.data();
    std::vector<u64> lines(HULL_LINES);
    HullDev h{};
    h.lines = lines.data();
    h.bidx = ids.data(); h.blist = ids.data(); h.bpos = pos.data(); h.bbox = box.data();
    for (int k = 0; k < nd; k++) {
        int p, q, r[64], w[64];
        if (fscanf(f, "%d %d", &p, &q) != 2) return 1;
        wave([&](int lane) { r[lane] = CALL_APEX; });
        wave([&](int lane) { w[lane] = CALL_NEAREST; });
        for (int l = 1; l < 64; l++)
            if (r[l] != r[0]) return 2;   // the wave's answer is one (of the nearest, lane 0's counts)
        printf("%d %d\n", r[0], w[0]);
    }
    printf("%d %lld\n", status, g_steps / 64);
    return 0;
}
"""


def _text(mesh):
    """The search, from the text of mesh.hip."""
    a = mesh.index("// The boundary vertices [b0, b1) of a set")
    b = mesh.index("// Creates the triangle (p, q, c) unless another demand did")
    return mesh[a:b]


@pytest.fixture(scope="module")
def search(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    d = tmp_path_factory.mktemp("hull")
    with open(os.path.join(CSRC, "dev_common.h")) as f:
        (d / "dev_common.h").write_text(f.read().replace("#define GA_INLINE __device__", "#define GA_INLINE __host__ __device__"))
    with open(os.path.join(CSRC, "kernels.h")) as f:
        (d / "kernels.h").write_text(f.read())
    with open(os.path.join(CSRC, "mesh.hip")) as f:
        (d / "hull.h").write_text(_text(f.read()))
    calls = ["-DCALL_APEX=hull_apex(m, h, p, q, hull_set(m, h, p), lane)",
             "-DCALL_NEAREST=hull_nearest(m, h, p, hull_set(m, h, p), lane)"]
    (d / "h.cpp").write_text(HARNESS)
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(d), str(d / "h.cpp"), "-o", str(d / "h")] +
                   calls, check=True, capture_output=True)

    def run(xy, demands, scale, other=0):
        (d / "in").write_text("%d %d %s %d\n" % (len(xy), len(demands), float(scale).hex(), other) +
                              "\n".join(float(x).hex() + " " + float(y).hex() for x, y in xy) + "\n" +
                              "\n".join("%d %d" % tuple(e) for e in demands) + "\n")
        out = subprocess.run([str(d / "h"), str(d / "in")], check=True, capture_output=True, text=True, timeout=30).stdout.split()
        r = [int(x) for x in out]
        assert r[-2] == 0   # no status
        return np.array(r[:-2]).reshape(-1, 2), r[-1]
    return run


def _morton(xy):
    q = ((xy - xy.min(0)) / max(np.ptp(xy), 1e-300) * 1023).astype(np.int64)
    key = np.zeros(len(xy), np.int64)
    for b in range(10):
        key |= ((q[:, 0] >> b & 1) << (2 * b + 1)) | ((q[:, 1] >> b & 1) << (2 * b))
    return xy[np.argsort(key, kind="stable")]


def _points(kind, n):
    rng = np.random.default_rng(n)
    a = rng.random(n) * 2 * np.pi
    if kind == "ring":
        r = 1 + 0.05 * rng.random(n)
    elif kind == "arc":
        a, r = a / 2, np.ones(n)
    elif kind == "box":
        return _morton(rng.random((n, 2)))
    elif kind == "sides":   # four straight sides, two of them sloped, and some points inside
        t = rng.permutation(4096)[:n] / 4096.0
        k = n // 5
        side = lambda i, a, b: np.array(a) + t[i * k:(i + 1) * k, None] * (np.array(b) - a)
        c = [(0.0, 0.0), (1.0, 0.25), (1.0, 1.25), (0.25, 1.25)]
        return _morton(np.concatenate([side(i, c[i], c[(i + 1) % 4]) for i in range(4)] + [0.25 + 0.5 * rng.random((n - 4 * k, 2))]))
    else:   # near the origin: distances down to 1e-13 of the largest
        r = 10.0 ** (-13 * rng.random(n))
    return _morton(np.stack([r * np.cos(a), r * np.sin(a)], 1))


def _demands(xy, k, seed):
    """Directed edges: to near vertices and to any."""
    rng = np.random.default_rng(seed)
    p = rng.integers(0, len(xy), k)
    q = np.array([rng.choice(np.argsort(((xy - xy[i]) ** 2).sum(1))[1:6]) if j % 4 else (i + 1 + rng.integers(len(xy) - 1)) % len(xy)
                  for j, i in enumerate(p)])
    return np.stack([p, q], 1)


def _scale(xy, T=512):
    return float(np.ptp(xy, axis=0).max()) / T


@pytest.mark.parametrize("kind", ["ring", "arc", "box", "origin", "sides"])
@pytest.mark.parametrize("e", [-365, 520])
def test_scaled(search, kind, e):
    xy = _points(kind, 1500)
    demands = _demands(xy, 120, 1)
    want, _ = search(xy, demands, _scale(xy))
    got, _ = search(np.ldexp(xy, e), demands, np.ldexp(_scale(xy), e))
    assert np.array_equal(got, want), (got != want).any(1).sum()


@pytest.mark.parametrize("e", [(-500, 500), (500, -500), (-1000, 100)])
def test_two_sets(search, e):
    """A box may hold vertices of two sets of a batch, of very different scale."""
    rng = np.random.default_rng(8)
    xy = np.stack(np.meshgrid(np.arange(38.0), np.arange(38.0)), -1).reshape(-1, 2) / 64
    xy = _morton(xy[rng.random(len(xy)) < 0.6])
    at = {tuple(v): k for k, v in enumerate(xy)}
    demands = []
    for k in range(120):   # axis-parallel edges of the lattice, the first box's vertices left of some
        for d in ((1, 0), (0, 1), (2, 0), (0, 2)):
            o = at.get((xy[k, 0] + d[0] / 64, xy[k, 1] + d[1] / 64))
            if o is not None:
                demands += [(k, o), (o, k)]
    demands = np.array(demands)
    want, _ = search(xy, demands, _scale(xy))
    other = 40
    got, _ = search(np.concatenate([np.ldexp(xy[:other], e[1]), np.ldexp(xy, e[0])]), demands + other, np.ldexp(_scale(xy), e[0]), other)
    assert np.array_equal(got[:, 0] - other * (got[:, 0] >= 0), want[:, 0])


def _apex(xy, p, q):
    """The vertex left of p -> q whose circle through p and q holds no other, in rationals."""
    F = [(Fraction(float(x)), Fraction(float(y))) for x, y in xy]
    (px, py), (qx, qy), best, at = F[p], F[q], None, []
    for i, (x, y) in enumerate(F):
        ax, ay, bx, by = px - x, py - y, qx - x, qy - y
        area = ax * by - ay * bx
        if area > 0:
            t = (ax * bx + ay * by) / area   # the cotangent of the angle under which it sees the edge
            if best is None or t < best:
                best, at = t, [i]
            elif t == best:
                at.append(i)   # on one circle with p and q
    return [-1] if best is None else at


@pytest.mark.parametrize("kind", ["ring", "arc", "origin", "sides"])
def test_rational(search, kind):
    xy = _points(kind, 700)
    demands = _demands(xy, 25, 2)
    got, _ = search(xy, demands, _scale(xy))
    for (p, q), (c, w) in zip(demands, got):
        assert c in _apex(xy, p, q)
        F = [(Fraction(float(x)) - Fraction(float(xy[p][0]))) ** 2 + (Fraction(float(y)) - Fraction(float(xy[p][1]))) ** 2
             for x, y in xy]
        assert w != p and F[w] == min(f for i, f in enumerate(F) if i != p)


@pytest.mark.parametrize("slope", [0.0, 0.25])
def test_straight_side(search, slope):
    """The hull edges along a straight side: after the first, no search looks along the whole side (190 boxes)."""
    rng = np.random.default_rng(4)
    n = 12000
    t = rng.permutation(16384)[:n] / 16384.0
    xy = _morton(np.concatenate([np.stack([t, slope * t], 1), [0, 1] + rng.random((500, 2))]))
    side = np.flatnonzero(xy[:, 1] == slope * xy[:, 0])
    side = side[np.argsort(xy[side, 0])]
    k = rng.integers(0, n - 1, 60)
    got, steps = search(xy, np.stack([side[k + 1], side[k]], 1), _scale(xy))
    assert (got[:, 0] == -1).all()
    assert steps < 2 * 190 + 60 * 25


@pytest.mark.gpu
@pytest.mark.parametrize("e", [-365, 520])
@pytest.mark.parametrize("kind", ["ring", "arc", "sides"])
def test_scaled_triangulation(kind, e):
    import galpha2d_amd as G
    print("case: scaled", kind, e, flush=True)
    if kind == "sides":   # two long straight sides, and points just outside
        t = np.random.default_rng(3).permutation(2048)[:700] / 2048.0
        xy = np.concatenate([np.stack([t, 0 * t], 1), np.stack([0.25 * t, 1 + 0.5 * t], 1), [[0.3, -0.001], [0.7, -0.002]]])
    else:
        xy = _points(kind, 1500)
    ctx = G.Context(0)
    want = ctx.delaunay(xy, 512)
    assert len(want) > 600
    assert np.array_equal(ctx.delaunay(np.ldexp(xy, e), 512), want)
    ctx.close()


@pytest.mark.gpu
def test_scaled_batch():
    """Sets of a batch with scales so far apart that a box of both overflows in either's."""
    import galpha2d_amd as G
    print("case: batch of scaled sets", flush=True)
    grid = np.stack(np.meshgrid(np.arange(20.0), np.arange(20.0)), -1).reshape(-1, 2)
    sets = [_points("ring", 700)[:650], grid, _points("arc", 500)[:333], grid[:390]]
    ctx = G.Context(0)
    want = ctx.batch(sets)
    for t, u in zip(ctx.batch([np.ldexp(xy, e) for xy, e in zip(sets, (-500, 480, 0, -360))]), want):
        assert len(u) > 300 and np.array_equal(t, u)
    ctx.close()
