"""Sites of the discrete diagram's pixels (k_splat, k_splat_own of pba.hip): the text of both kernels on the
host, the threads of the second one in orders that a GPU may run them in.  A pixel's site is its point
of the smallest input index, stored as its own (renumbered) index, whatever the order."""
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(__file__), "..", "galpha2d_amd", "csrc")
HIPCC = "/opt/rocm/bin/hipcc"
HARNESS = r"""
#include <hip/hip_runtime.h>
#include <cmath>
#include <cstdio>
#include <vector>
#include "dev_common.h"
#include "kernels.h"
static struct { int x; } h_block, h_dim{1}, h_thread;
#define blockIdx h_block
#define blockDim h_dim
#define threadIdx h_thread
#define atomicMin(p, v) (*(p) = *(p) < (v) ? *(p) : (v))
#undef GA_INLINE
#define GA_INLINE static inline
#undef __global__
#define __global__ static
#include "splat.h"
// n, number of cells, for every own index its input index and cell, then the threads of k_splat_own
// in their order; prints the site of every cell
int main()
{
    int n, nc;
    while (scanf("%d %d", &n, &nc) == 2) {
        const int T = 64;
        std::vector<int> perm(n), order(n), vset(n, 0), pix(n), smap(T * T, 0x7fffffff);
        std::vector<double2> xy(n);
        for (int i = 0; i < n; i++) {
            int c;
            if (scanf("%d %d", &perm[i], &c) != 2) return 1;
            xy[i] = make_double2(c + 0.5, 3.5);
        }
        for (int i = 0; i < n; i++)
            if (scanf("%d", &order[i]) != 1) return 1;
        SetDesc sd{};
        sd.logT = 6; sd.n = n; sd.inv = sd.scale = 1.0; sd.margin = 5;
        BatchDev b{};
        b.sets = &sd; b.nsets = 1; b.vset = vset.data(); b.ntot = b.V = n;
        for (h_block.x = 0; h_block.x < n; h_block.x++) k_splat(xy.data(), b, perm.data(), smap.data(), pix.data());
        for (int i : order) {
            h_block.x = i;
            k_splat_own(b, perm.data(), nullptr, pix.data(), smap.data());
        }
        for (int c = 0; c < nc; c++) printf("%d ", smap[(c + 5) * T + 8]);
        printf("\n");
    }
    return 0;
}
"""


def test_every_order(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not installed")
    for name in ("dev_common.h", "kernels.h"):
        with open(os.path.join(CSRC, name)) as f:
            (tmp_path / name).write_text(f.read().replace("#define GA_INLINE __device__", "#define GA_INLINE __host__ __device__"))
    with open(os.path.join(CSRC, "pba.hip")) as f:
        text = f.read()
    pixel = text[text.index("// pixel of a real point in its set's texture"):text.index("// Spatial order of the real points")]
    splat = text[text.index("// Map real points to pixels"):text.index("// ---- phase 1")]
    (tmp_path / "splat.h").write_text(pixel + splat)
    (tmp_path / "s.cpp").write_text(HARNESS)
    subprocess.run([HIPCC, "--offload-host-only", "-O1", "-std=c++17", "-I", str(tmp_path), str(tmp_path / "s.cpp"), "-o",
                    str(tmp_path / "s")], check=True, capture_output=True)
    text, want = "", []
    for seed in range(200):
        rng = np.random.default_rng(seed)
        n, nc = int(rng.integers(2, 60)), int(rng.integers(1, 5))
        cell = np.sort(rng.integers(0, nc, n))           # own indices go by cells
        perm = np.arange(n) if seed % 3 == 0 else rng.permutation(n) if seed % 3 == 1 else np.roll(np.arange(n), seed % 7)
        win = [min(np.flatnonzero(cell == c), key=lambda i: perm[i], default=0x7fffffff) for c in range(nc)]
        order = [i for i in win if i < n] + [i for i in rng.permutation(n) if i not in win]   # the winners store first
        if seed % 2:
            order = rng.permutation(n)
        text += "%d %d\n" % (n, nc) + "\n".join("%d %d" % x for x in zip(perm, cell)) + "\n" + " ".join(map(str, order)) + "\n"
        want.append(win)
    out = subprocess.run([str(tmp_path / "s")], input=text, check=True, capture_output=True, text=True).stdout.splitlines()
    assert [[int(x) for x in line.split()] for line in out] == want
