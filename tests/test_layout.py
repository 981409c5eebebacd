"""LDS layouts of the host planner: budgets that hold a system, and regions that hold what the
kernels put there.  Host code of csrc/stc_internal.h, compiled by itself."""
import os
import subprocess

import pytest

from staccato_amd import build

MAIN = r'''
#include <cstdio>
#include "stc_internal.h"
using namespace stc;
int main() {
    int kind, ts, n, nrhs, budget, jb, adj;
    while (scanf("%d %d %d %d %d %d %d", &kind, &ts, &n, &nrhs, &budget, &jb, &adj) == 7) {
        int maxr = 2;
        while (64 * maxr < n) maxr *= 2;
        const Layout L = kind == 1 ? plan_layout(n, nrhs, ts, budget, jb, adj, maxr)
                                   : plan_layout_wide(n, nrhs, ts, budget, jb, adj, maxr);
        const int waves = sweep_threads(ts == 8, maxr, kind == 1 ? 0 : 1) / 64;
        printf("%d %d %d %d %d %d %d\n", L.lds <= budget, L.small, L.jb, L.G, L.lds, waves, lds_fixed_bytes(n, waves));
    }
}
'''


def _layouts(tmp_path, cases):
    src, exe = tmp_path / "layout.cpp", tmp_path / "layout"
    src.write_text(MAIN)
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(build.hipcc())))
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I" + build.CSRC,
                    "-I" + os.path.join(rocm, "include"), "-o", str(exe), str(src)], check=True)
    out = subprocess.run([str(exe)], input="\n".join(" ".join(map(str, c)) for c in cases),
                         capture_output=True, text=True, check=True).stdout
    return [tuple(map(int, line.split())) for line in out.splitlines()]


@pytest.mark.parametrize("case,small,jb,G", [
    # kind (1 register panel, 2 wide), bytes an element, n, nrhs, budget, jb cap, adjoint
    ((1, 8, 143, 1, 16384, 4, 0), 0, 4, 1),
    ((1, 8, 230, 1, 20480, 16, 0), 0, 4, 1),
    ((1, 8, 512, 4, 53 * 1024, 16, 0), 0, 8, 2),
    ((1, 16, 29, 1, 16384, 4, 0), 1, 0, 1),
    ((1, 16, 657, 4, 53 * 1024, 4, 0), 0, 4, 1),
    ((1, 16, 909, 1, 80 * 1024, 4, 1), None, None, None),   # beyond it either way
    ((2, 8, 74, 1, 16384, 32, 0), 0, 16, 1),
    ((2, 8, 843, 4, 120000, 32, 0), 0, 16, 4),
    ((2, 16, 99, 1, 160 * 1024 - 256, 16, 0), 1, 0, 1),
])
def test_budgets(tmp_path, case, small, jb, G):
    """The reduction scratch is that of the kernel's own wavefronts, and the eight-wavefront
    kernels' larger pivot-candidate buffers lie where the inverted blocks come later."""
    ok, s, j, g = _layouts(tmp_path, [case])[0][:4]
    if jb is None:
        assert not ok
    else:
        assert ok and (s, j, g) == (small, jb, G)


def test_wide_regions(tmp_path):
    """Panel, inverted blocks or pivot candidates, moved rows, and the two U blocks of the
    left-looking update fit the launch's LDS at every order, next to the fixed region."""
    cases = [(2, ts, n, 1, b, 32, adj) for ts in (8, 16) for n in range(1, 1025) for adj in (0, 1)
             for b in (16384, 20480, 24576, 40960, 80 * 1024, 160 * 1024 - 256)]
    some = 0
    for c, (ok, small, jb, G, lds, waves, fixed) in zip(cases, _layouts(tmp_path, cases)):
        if not ok or small:
            continue
        ts, n = c[1], c[2]
        cols = 32 if ts == 8 else 16
        panel = (n | 1) * jb * ts
        assert panel + max(jb * 16 * ts, 2 * waves * (16 * ts + 16)) + 256 <= lds - fixed, c
        assert 2 * cols * 17 * ts <= lds - fixed, c
        some += 1
    assert some > 5000
