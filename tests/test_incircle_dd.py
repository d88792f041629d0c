"""Incircle sign in pairs of doubles (incircle_dd), built for the host from the device header, against
rationals: it must be right wherever it decides, and decide what lies a few last places off a circle."""
import math
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
    double v[9];
    while (scanf("%la %la %la %la %la %la %la %la %la", v, v + 1, v + 2, v + 3, v + 4, v + 5, v + 6, v + 7, v + 8) == 9)
        printf("%d\n", incircle_dd(make_double2(v[0], v[1]), make_double2(v[2], v[3]), make_double2(v[4], v[5]),
                                   make_double2(v[6], v[7]), v[8]));
    return 0;
}
"""


def _cases(kind, n=800):
    """Four points and the power of two for their differences."""
    rng = random.Random(kind)
    for _ in range(n):
        e = 0
        if kind in ("circle", "far", "scaled"):
            a = [rng.uniform(0, 7) for _ in range(4)]
            cx, cy = (rng.uniform(-1, 1) * 2.0 ** 12, 1.5) if kind == "far" else (0.0, 0.0)
            v = [c for t in a for c in (cx + math.cos(t), cy + math.sin(t))]
            if kind == "scaled":
                e = rng.choice([-365, -800, 480, 900])
                v = [math.ldexp(x, e) for x in v]
        elif kind == "lattice":   # many exactly on one circle
            v = [rng.randint(-6, 6) * 0.5 for _ in range(8)]
        elif kind == "wide":      # differences of very different sizes
            v = [rng.choice([-1, 1]) * rng.random() * 2.0 ** -rng.choice([0, 10, 30, 60, 200]) for _ in range(8)]
        else:                     # two last places off the corners of a square
            v = [x * (1 + rng.randint(-2, 2) * 2.0 ** -52) for x in (0.7, 0.7, -0.7, 0.7, -0.7, -0.7, 0.7, -0.7)]
        yield v + [2.0 ** -e]


@pytest.mark.parametrize("kind", ["circle", "far", "scaled", "lattice", "wide", "square"])
def test_incircle_dd(kind, tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    with open(os.path.join(CSRC, "dev_common.h")) as f:
        hdr = f.read().replace("#define GA_INLINE __device__", "#define GA_INLINE __host__ __device__")
    (tmp_path / "dev_common.h").write_text(hdr)
    (tmp_path / "o.cpp").write_text(HARNESS)
    subprocess.run([HIPCC, "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(tmp_path),
                    str(tmp_path / "o.cpp"), "-o", str(tmp_path / "o")], check=True, capture_output=True)
    cases = list(_cases(kind))
    text = "\n".join(" ".join(x.hex() for x in v) for v in cases)
    out = subprocess.run([str(tmp_path / "o")], input=text, check=True, capture_output=True, text=True).stdout.split()
    assert len(out) == len(cases)
    decided = 0
    for v, r in zip(cases, map(int, out)):
        f = [Fraction(x) for x in v[:8]]
        x, y = [f[2 * k] - f[6] for k in range(3)], [f[2 * k + 1] - f[7] for k in range(3)]
        det = sum((x[k] ** 2 + y[k] ** 2) * (x[(k + 1) % 3] * y[(k + 2) % 3] - x[(k + 2) % 3] * y[(k + 1) % 3]) for k in range(3))
        assert r in ((det > 0) - (det < 0), 0), v
        decided += r != 0 or det == 0
    # square: the sum of eight last-place steps of -2 .. 2 is zero in 10% of the cases, and what is left then is
    # below the bound
    assert decided > {"wide": 0.3, "square": 0.85}.get(kind, 0.95) * len(cases)
