"""Exact orientation from exact differences (orient_diff), built for the host from the device header, against
rationals: points of few bits and their collinear triples, last-place neighbours, zeros, ends of the range.  It
answers 2 where a difference or a product is not exact, and never on a lattice."""
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
    while (scanf("%la %la %la %la %la %la", v, v + 1, v + 2, v + 3, v + 4, v + 5) == 6)
        printf("%d\n", orient_diff(make_double2(v[0], v[1]), make_double2(v[2], v[3]), make_double2(v[4], v[5])));
    return 0;
}
"""


def _cases(kind, n=600):
    rng = random.Random(kind)
    for _ in range(n):
        if kind == "lattice":
            v = [rng.randint(-40, 40) / 16.0 for _ in range(6)]
        elif kind == "line":      # 26-bit multiples of one direction
            d = rng.choice([(1.0, 0.375), (0.5, -1.25), (3.0, 7.0)])
            v = [c * k for k in (rng.randint(0, 1 << 26) * 2.0 ** -26 for _ in range(3)) for c in d]
        elif kind == "near":      # collinear but for one last place
            v = [0.5, 0.5, 12.0, 12.0, 24.0, 24.0]
            v = [x + rng.randint(-2, 2) * 2.0 ** -rng.choice([48, 49, 52, 53]) for x in v]
        else:
            s = rng.choice([2.0 ** -520, 2.0 ** -466, 2.0 ** 490, 2.0 ** 520])
            v = [s * rng.choice([0.0, 1.0, -1.0, 0.75, rng.random()]) for _ in range(6)]
        yield v


@pytest.mark.parametrize("kind", ["lattice", "line", "near", "ends"])
def test_orient_diff(kind, tmp_path):
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
    seen = set()
    for v, r in zip(cases, map(int, out)):
        ax, ay, bx, by, cx, cy = (Fraction(x) for x in v)
        d = (ax - cx) * (by - cy) - (ay - cy) * (bx - cx)
        assert r in ((d > 0) - (d < 0), 2), v
        seen.add(r)
    assert seen >= ({0} if kind == "line" else {-1, 0, 1})
    assert 2 not in seen or kind in ("near", "ends")
