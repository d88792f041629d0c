"""The floating-point filters of the two predicates, built for the host from the device header, against rationals on
coordinates whose products underflow: they must be right or leave the sign open."""
import os
import random
import subprocess
from fractions import Fraction

import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "galpha2d_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"
HARNESS = r"""
#include <hip/hip_runtime.h>
#include <cstdio>
#include "dev_common.h"
int main()
{
    double v[8];
    while (scanf("%la %la %la %la %la %la %la %la", v, v + 1, v + 2, v + 3, v + 4, v + 5, v + 6, v + 7) == 8) {
        const double2 a = make_double2(v[0], v[1]), b = make_double2(v[2], v[3]), c = make_double2(v[4], v[5]),
                      d = make_double2(v[6], v[7]);
        printf("%d %d\n", orient_filter(a, b, c), incircle_filter(a, b, c, d));
    }
    return 0;
}
"""


def _cases(kind, scales, n=3000):
    rng = random.Random(kind)
    for _ in range(n):
        s = 2.0 ** rng.choice(scales)
        if kind == "random":
            v = [rng.uniform(-1, 1) for _ in range(8)]
        elif kind == "near":    # almost collinear and almost on one circle
            v = [x * (1 + rng.randint(-3, 3) * 2.0 ** -50) for x in (0.7, 0.7, -0.7, 0.7, -0.7, -0.7, 0.7, -0.7)]
            v[2:6] = rng.choice([v[2:6], [0.35 * (1 + 2.0 ** -52), 0.35, 0.1, 0.1]])
        else:                   # far and close points together
            v = [rng.uniform(-1, 1) * 2.0 ** -rng.choice([0, 0, 5, 40]) for _ in range(8)]
        yield [x * s for x in v]


@pytest.mark.parametrize("kind", ["random", "near", "mixed"])
@pytest.mark.parametrize("scales", [(-250, -262, -265, -266, -267, -268, -269, -270), (-500, -530, -534, -536, -537, -538), (0, -100, -200)],
                         ids=["incircle", "orient", "ordinary"])
def test_filters(kind, scales, tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    with open(os.path.join(CSRC, "dev_common.h")) as f:
        hdr = f.read().replace("#define GA_INLINE __device__", "#define GA_INLINE __host__ __device__")
    (tmp_path / "dev_common.h").write_text(hdr)
    (tmp_path / "o.cpp").write_text(HARNESS)
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(tmp_path),
                    str(tmp_path / "o.cpp"), "-o", str(tmp_path / "o")], check=True, capture_output=True)
    cases = list(_cases(kind, scales))
    text = "\n".join(" ".join(x.hex() for x in v) for v in cases)
    out = subprocess.run([str(tmp_path / "o")], input=text, check=True, capture_output=True, text=True).stdout.split()
    assert len(out) == 2 * len(cases)
    decided = 0
    for v, o, i in zip(cases, map(int, out[::2]), map(int, out[1::2])):
        f = [Fraction(x) for x in v]
        det = (f[0] - f[4]) * (f[3] - f[5]) - (f[1] - f[5]) * (f[2] - f[4])
        assert o in ((det > 0) - (det < 0), 0), v
        x, y = [f[2 * k] - f[6] for k in range(3)], [f[2 * k + 1] - f[7] for k in range(3)]
        det = sum((x[k] ** 2 + y[k] ** 2) * (x[(k + 1) % 3] * y[(k + 2) % 3] - x[(k + 2) % 3] * y[(k + 1) % 3]) for k in range(3))
        assert i in ((det > 0) - (det < 0), 0), v
        decided += o != 0 and i != 0
    if scales[0] == 0 and kind == "random":
        assert decided > 0.99 * len(cases)   # what the filters are for


@pytest.mark.gpu
@pytest.mark.parametrize("e", [-240, -250, -262, -267, -535])
def test_triangulation(e):
    import numpy as np
    import galpha2d_amd as G
    from galpha2d_amd import datagen
    print("case: scaled by 2 to the", e, flush=True)
    ctx = G.Context(0)
    for xy, T in ((datagen.uniform(3, 3000), 512), (datagen.gaussian_clusters(np.random.default_rng(1), 3000, 8, 0.01), 512),
                  (datagen.lattice_clusters(3000, side=54, nclusters=8), 512)):
        assert np.array_equal(ctx.delaunay(np.ldexp(xy, e), T), ctx.delaunay(xy, T))
    ctx.close()
