"""Performance cases: the calls that users of galpha2d_amd make, over the sizes they make them at.

Kinds of call (`kind` of a case):
  alpha_host    compute_alpha_shapes(): host points in, host triangles and the whole alpha result out
  dt_host       gpudt_compute_dt() with constraint edges: host arrays in and out
  dt_noalloc    compute_device_noalloc(): device points in, triangles into the caller's device buffer
  dt_device     Context.compute_device(): device points in, triangles left on the device
  alpha_device  Context.compute_device(with_alpha=True), then the alpha complex at one alpha value
                (rank lookup and the classes of all vertices, edges and triangles, on the device)
  batch_device  Context.batch_device(with_alpha=True): many device sets in one pass, triangles on the device
  batch_host    Context.batch(): many host sets in one pass, host triangles out
  serve         Server: a burst of requests, every request's triangles and alpha result to the host

The number of triangles, edges and spectrum values depends on the points, so results go to arrays of
the caller's that hold the most there can be (2 n triangles, 3 n edges), zero past the end.
"""
import math

import numpy as np
import torch

import galpha2d_amd as G
from galpha2d_amd import datagen


def listed():
    return [
        # one small set through the reference-named call, host to host: the smallest call (latency)
        dict(name="alpha_host_1k", kind="alpha_host", n=1000, texture=512, dist="uniform"),
        # a clustered set of an odd, ordinary size, host to host
        dict(name="alpha_host_12k_clusters", kind="alpha_host", n=12007, texture=512, dist="clusters"),
        # a triangulation inside a loop that must not allocate
        dict(name="dt_noalloc_5k", kind="dt_noalloc", n=5000, texture=512, dist="uniform"),
        # a triangulation of a device-resident set just past a power of two
        dict(name="dt_device_65k", kind="dt_device", n=65537, texture=1024, dist="uniform"),
        # an ordinary alpha shape of a device-resident clustered set, then one query
        dict(name="alpha_device_250k_clusters", kind="alpha_device", n=250001, texture=2048, dist="clusters"),
        # the plain method at scale: the benchmark's headline workload, then one query
        dict(name="alpha_device_1m", kind="alpha_device", n=1048576, texture=4096, dist="uniform"),
        # the degenerate stress workload: half a lattice (co-circular quadruples), half clusters
        dict(name="alpha_device_2m_lattice", kind="alpha_device", n=2000000, texture=8192, dist="lattice"),
        # a large triangulation without the alpha spectrum
        dict(name="dt_device_4m", kind="dt_device", n=4000000, texture=8192, dist="uniform"),
        # a constrained triangulation (one polygon in each cell of a grid), host to host
        dict(name="cdt_host_100k", kind="dt_host", n=100000, texture=2048, dist="uniform", cells=42, per=6),
        # a quarter of the benchmark's batch of sets: throughput
        dict(name="batch_device_1024", kind="batch_device", sets=1024, lo=256, hi=65536),
        # a few dozen small host sets triangulated in one call
        dict(name="batch_host_48", kind="batch_host", sets=48, lo=256, hi=16384),
        # a burst of serving requests on four slots
        dict(name="serve_16", kind="serve", sets=16, lo=1000, hi=100000),
    ]


def draw(rng):
    def size(lo, hi):
        return int(math.exp(rng.uniform(math.log(lo), math.log(hi))))

    kind = rng.choice(["alpha_host", "dt_host", "dt_noalloc", "dt_device", "alpha_device", "alpha_device",
                       "batch_device", "batch_host", "serve"])
    case = dict(kind=kind)
    if kind == "batch_device":
        case.update(sets=size(8, 800), lo=256, hi=size(2048, 65536))
    elif kind == "batch_host":
        case.update(sets=size(4, 60), lo=rng.choice([64, 256, 1000]), hi=size(2048, 32768))
    elif kind == "serve":
        case.update(sets=size(2, 24), lo=1000, hi=size(5000, 200000))
    else:
        top = dict(alpha_host=100000, dt_host=200000, dt_noalloc=65536, dt_device=4000000, alpha_device=2000000)[kind]
        n = size(300, top)
        texture = G.auto_texture(n)
        if kind != "dt_noalloc" and texture < 4096 and rng.random() < 0.25:
            texture *= 2
        dist = "uniform" if kind == "dt_host" else rng.choice(["uniform", "uniform", "clusters", "lattice"])
        case.update(n=n, texture=texture, dist=dist)
        if kind == "dt_host":
            case.update(cells=max(2, int(math.sqrt(n / rng.uniform(20, 120)))), per=rng.randint(3, 8))
    return case


def _points(dist, n, seed):
    if dist == "uniform":
        return datagen.uniform(seed, n)
    if dist == "clusters":
        return datagen.gaussian_clusters(np.random.default_rng(seed), n, 8, 0.01)
    return datagen.lattice_clusters(n, side=max(2, math.isqrt(n)), seed=seed)


def _cell_polygons(xy, cells, per):
    """One star polygon of up to `per` points in each cell of a cells x cells grid, as constraint
    pairs: edges stay inside their convex cell and go round its points' centre, so none cross."""
    ij = np.minimum((xy * cells).astype(np.int64), cells - 1)
    key = ij[:, 0] * cells + ij[:, 1]
    order = np.argsort(key, kind="stable")
    k = key[order]
    first = np.searchsorted(k, k, side="left")
    take = order[np.arange(len(k)) - first < per]          # the first `per` points of each cell
    k = key[take]
    start = np.searchsorted(k, k, side="left")
    count = np.searchsorted(k, k, side="right") - start
    _, inv = np.unique(k, return_inverse=True)
    centre = np.stack([np.bincount(inv, xy[take, a]) for a in (0, 1)], 1) / np.bincount(inv)[:, None]
    d = xy[take] - centre[inv]
    take = take[np.lexsort((np.arctan2(d[:, 1], d[:, 0]), k))]
    pos = np.arange(len(k))
    nxt = np.where(pos + 1 < start + count, pos + 1, start)
    keep = count >= 3
    return np.stack([take[keep], take[nxt[keep]]], 1).astype(np.int32)


def _alpha_value(n):
    """A squared radius in the middle of the spectrum of n points spread over the unit square."""
    return 0.4 / n


def _sizes(case):
    """Set sizes of a case with many sets, log-uniform in [lo, hi]: the case's own, whatever the seed."""
    rng = np.random.default_rng(case["sets"])
    return np.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"]), case["sets"])).astype(np.int64)


# the most entries that an alpha result array of n points has
ALPHA_ROOM = dict(spectrum=5, tri_ro_rank=2, edge_t=3, edge_vopp=3, edge_ro_rank=3, edge_nu_min=3, edge_nu_max=3,
                  vert_nu_min=1, vert_nu_max=1, master_simplex=13, master_st=13, master_at=13, spec_pointers=5)


def _host_room(n, sets, alpha):
    room = {"triangles": np.zeros((2 * n, 9), np.int32)}
    if alpha:
        room["alpha"] = {k: np.zeros(m * n + sets, np.float64 if k == "spectrum" else np.int32)
                         for k, m in ALPHA_ROOM.items()}
    return room


def prepare(case, seed):
    kind = case["kind"]
    state = dict(case)
    if "sets" in case:
        sizes = _sizes(case)
        state["total"] = int(sizes.sum())
    if kind in ("batch_device", "batch_host"):
        # half uniform, half Gaussian clusters, as the batched benchmark makes them
        sets = [_points("clusters" if i % 2 else "uniform", int(n), seed * 1000003 + i) for i, n in enumerate(sizes)]
        state["ctx"] = G.Context(0)
        if kind == "batch_host":
            state["xy"] = sets
            state["room"] = _host_room(state["total"], len(sets), False)
        else:
            state["offsets"] = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
            state["xy"] = torch.from_numpy(np.concatenate(sets)).cuda()
            state["room"] = torch.zeros((2 * state["total"], 9), dtype=torch.int32, device="cuda")
        return state
    if kind == "serve":
        # windows of one pool, as the serving benchmark cuts them; four slots, resident buffers
        pool = datagen.uniform(seed, case["hi"] + 1)
        starts = np.random.default_rng(seed).integers(0, len(pool) - sizes + 1)
        state["xy"] = [pool[s:s + n].copy() for s, n in zip(starts, sizes)]
        state["server"] = G.Server(0, slots=4, hbm_budget_bytes=32 << 30, max_group=64, max_group_points=2000000)
        state["room"] = _host_room(state["total"], len(sizes), True)
        return state
    n = case["n"]
    xy = _points(case["dist"], n, seed)
    if kind in ("alpha_host", "dt_host"):
        state["xy"] = xy
        state["room"] = _host_room(n, 1, kind == "alpha_host")
        if kind == "dt_host":
            state["constraints"] = _cell_polygons(xy, case["cells"], case["per"])
        return state
    state["xy"] = torch.from_numpy(xy).cuda()
    state["room"] = torch.zeros((2 * n, 9), dtype=torch.int32, device="cuda")
    if kind != "dt_noalloc":
        state["ctx"] = G.Context(0)
    if kind == "alpha_device":
        state["classes"] = [torch.zeros(k * n, dtype=torch.uint8, device="cuda") for k in (1, 3, 2)]
    return state


class _DeviceArray:
    def __init__(self, ptr, shape):
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, typestr="<i4", version=2)


def _keep_device_triangles(ctx, room):
    """Copies the triangles that the context left on the device into the caller's tensor."""
    p, n = G.C.c_void_p(), G.C.c_int()
    G.lib().galphaDeviceTriangles(ctx._h, G.C.byref(p), G.C.byref(n))
    room[:n.value].copy_(torch.as_tensor(_DeviceArray(p.value, (n.value, 9)), device="cuda"))


def _keep(room, results):
    """Stores host results (triangles, alpha result or None) one after another."""
    end = dict.fromkeys(ALPHA_ROOM, 0)
    at = 0
    for tris, alpha in results:
        room["triangles"][at:at + len(tris)] = tris
        at += len(tris)
        for k, a in (alpha or {}).items():
            room["alpha"][k][end[k]:end[k] + len(a)] = a
            end[k] += len(a)
    return dict(room, counts=[at] + list(end.values()))


def run(state):
    kind, room = state["kind"], state["room"]
    if kind == "alpha_host":
        return _keep(room, [G.compute_alpha_shapes(state["xy"], state["texture"])])
    if kind == "dt_host":
        return _keep(room, [(G.gpudt_compute_dt(state["xy"], state["texture"], state["constraints"]), None)])
    if kind == "batch_host":
        return _keep(room, [(tris, None) for tris in state["ctx"].batch(state["xy"])])
    if kind == "serve":
        server = state["server"]
        tickets = [server.submit(x) for x in state["xy"]]

        def finished(ticket):
            server.wait(ticket)
            return server.result(ticket)
        return _keep(room, map(finished, tickets))
    xy = state["xy"]
    if kind == "dt_noalloc":
        count = G.compute_device_noalloc(xy.data_ptr(), state["n"], state["texture"], room.data_ptr(), len(room))
        return {"triangles": room, "count": count}
    ctx = state["ctx"]
    if kind == "batch_device":
        count = ctx.batch_device(xy.data_ptr(), state["offsets"], with_alpha=True)
    else:
        count = ctx.compute_device(xy.data_ptr(), state["n"], state["texture"], with_alpha=kind == "alpha_device")
    _keep_device_triangles(ctx, room)
    out = {"triangles": room, "count": count}
    if kind == "alpha_device":
        vert, edge, tri = state["classes"]
        rank = ctx.alpha_rank(_alpha_value(state["n"]))
        if G.lib().galphaClassifyDevice(ctx._h, rank, vert.data_ptr(), edge.data_ptr(), tri.data_ptr(), None) < 0:
            raise G.GalphaError("galphaClassifyDevice failed")
        out.update(rank=rank, vertex_classes=vert, edge_classes=edge, triangle_classes=tri)
    return out


def work(case):
    """Points (16 B) read once; triangles (2 n of 36 B) written once; with the alpha result its arrays
    too: spectrum (4 n of 8 B), ranks and intervals of triangles, edges and vertices (76 n B), master
    list (12 n entries of 12 B) and rank pointers (16 n B).  Arithmetic: one orientation and one
    incircle test per triangle and edge, one radius and one attachment test per simplex."""
    kind = case["kind"]
    n = case["n"] if "n" in case else int(_sizes(case).sum())
    size, flops = 16 + 72, 2 * 15 + 3 * 50
    if "alpha" in kind or kind in ("serve", "batch_device"):
        size += 32 + 76 + 144 + 16
        flops += 2 * 40 + 3 * 30
    if kind == "alpha_device":
        size += 6
    return {"bytes": float(size) * n, "flops": float(flops) * n}


def _delaunay(p):
    """Delaunay triangles of points in general position, by gift wrapping: across each directed
    edge, the point to its left that sees it under the largest angle."""
    x, y = p[:, 0], p[:, 1]
    a = int(np.lexsort((x, y))[0])
    d = p - p[a]
    with np.errstate(all="ignore"):
        ang = np.arctan2(d[:, 1], d[:, 0])
    ang[a] = np.inf
    todo, done, out = [(a, int(np.argmin(ang)))], set(), []
    while todo:
        e = todo.pop()
        if e in done:
            continue
        a, b = e
        ax, ay, bx, by = x[a] - x, y[a] - y, x[b] - x, y[b] - y
        area = ax * by - ay * bx                       # twice the area of (a, b, c), seen from c
        area[a] = area[b] = 0.0
        left = np.nonzero(area > 0)[0]
        if not len(left):
            continue
        c = int(left[np.argmin((ax[left] * bx[left] + ay[left] * by[left]) / area[left])])
        out.append((a, b, c))
        done.update(((a, b), (b, c), (c, a)))
        todo += [(b, a), (c, b), (a, c)]
    return np.array(out)


def exact(case, seed):
    """The spectrum in plain numpy; everything else that the cases return is whole numbers.  None for
    sets that take too long that way, and for lattices, where equal values decide the spectrum."""
    if case["kind"] != "alpha_host" or case["n"] > 20000 or case["dist"] == "lattice":
        return None
    p = _points(case["dist"], case["n"], seed)
    t = _delaunay(p)
    a, b, c = p[t[:, 0]], p[t[:, 1]], p[t[:, 2]]

    def sq(u, v):
        return ((u - v) ** 2).sum(1)

    area = (b[:, 0] - a[:, 0]) * (c[:, 1] - a[:, 1]) - (b[:, 1] - a[:, 1]) * (c[:, 0] - a[:, 0])
    values = [np.zeros(1), sq(a, b) * sq(b, c) * sq(c, a) / (4 * area * area)]
    # an edge counts unless the circle on it as diameter holds an apex
    ends = np.concatenate([t[:, [0, 1]], t[:, [1, 2]], t[:, [2, 0]]])
    apex = p[np.concatenate([t[:, 2], t[:, 0], t[:, 1]])]
    u, v = p[ends[:, 0]], p[ends[:, 1]]
    attached = ((u - apex) * (v - apex)).sum(1) <= 0
    key, inv = np.unique(np.sort(ends, 1) @ np.array([len(p), 1]), return_inverse=True)
    free = np.bincount(inv, attached) == 0
    values.append(sq(p[key[free] // len(p)], p[key[free] % len(p)]) / 4)
    spectrum = np.zeros(ALPHA_ROOM["spectrum"] * len(p) + 1)
    values = np.sort(np.concatenate(values))
    spectrum[:len(values)] = values
    return {"triangles": None, "counts": [None] * (1 + len(ALPHA_ROOM)),
            "alpha": dict(dict.fromkeys(ALPHA_ROOM), spectrum=spectrum)}
