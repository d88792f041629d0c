"""Exact orientation by floating-point expansions (orient_exact up to a spread of 2^60) and by big
integers beyond, built for the host from the device header, against rationals: points on a line moved
by single units in the last place, coordinates on either side of the spread limit, and zeros."""
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
    double v[6];
    while (scanf("%la %la %la %la %la %la", v, v + 1, v + 2, v + 3, v + 4, v + 5) == 6) {
        int ovf = 0;
        const int r = orient_exact(make_double2(v[0], v[1]), make_double2(v[2], v[3]), make_double2(v[4], v[5]), &ovf);
        printf("%d %d\n", r, ovf);
    }
    return 0;
}
"""


def _step(x, k):
    import numpy as np
    for _ in range(abs(k)):
        x = float(np.nextafter(x, np.inf if k > 0 else -np.inf))
    return x


def _cases(kind, n=400):
    rng = random.Random(kind)
    for _ in range(n):
        if kind == "line":
            s, t = rng.uniform(-3, 3), [rng.uniform(0.1, 1) for _ in range(3)]
            v = [c for x in t for c in (x, _step(s * x, rng.randint(-1, 1)))]
        elif kind == "spread":   # smallest and largest coordinate 2^57 to 2^63 apart
            e = rng.randint(57, 63)
            v = [rng.choice([1.0, 2.0 ** -e, 1.5 * 2.0 ** -e, -1.0, 2.0 ** -(e // 2)]) for _ in range(6)]
        elif kind == "zeros":
            v = [rng.choice([0.0, 0.0, 1.0, -1.0, rng.random()]) for _ in range(6)]
        else:                    # near the ends of the range of the products
            s = rng.choice([2.0 ** -431, 2.0 ** 431])
            v = [s * (1 + rng.random()) * rng.choice([1, -1]) for _ in range(6)]
            if rng.random() < 0.5:
                v[4:] = [v[0] + 2 * (v[2] - v[0]), v[1] + 2 * (v[3] - v[1])]
        yield v


@pytest.mark.parametrize("kind", ["line", "spread", "zeros", "ends"])
def test_orient_exact(kind, tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    with open(os.path.join(CSRC, "dev_common.h")) as f:
        hdr = f.read().replace("#define GA_INLINE __device__", "#define GA_INLINE __host__ __device__")
    (tmp_path / "dev_common.h").write_text(hdr)
    (tmp_path / "o.cpp").write_text(HARNESS)
    subprocess.run([HIPCC, "-O2", "-std=c++17", "-ffp-contract=off", "-I", str(tmp_path), str(tmp_path / "o.cpp"), "-o",
                    str(tmp_path / "o")], check=True, capture_output=True)
    cases = list(_cases(kind))
    text = "\n".join(" ".join(x.hex() for x in v) for v in cases)
    out = subprocess.run([str(tmp_path / "o")], input=text, check=True, capture_output=True, text=True).stdout.split()
    assert len(out) == 2 * len(cases)
    signs = set()
    for v, r, ovf in zip(cases, out[::2], out[1::2]):
        ax, ay, bx, by, cx, cy = (Fraction(x) for x in v)
        d = (ax - cx) * (by - cy) - (ay - cy) * (bx - cx)
        want = (d > 0) - (d < 0)
        assert (int(r), int(ovf)) == (want, 0), v
        signs.add(want)
    assert signs >= {-1, 1}
