"""The GEMM planner's choices, on the CPU: a small driver linked with the library asks for the kernel
of one GEMM per line."""
import os
import subprocess

import pytest

from conftest import PKG

DRIVER = r"""
#include "sdu_internal.h"
#include <cstdio>
using namespace sdu;
int main() {
    static double st;
    int M, N, K, hw;
    while (scanf("%d %d %d %d", &M, &N, &K, &hw) == 4) {
        GemmArgs g{};
        g.amode = A_DENSE;
        g.M = M; g.N = N; g.K = K;
        g.lda = g.K1 = K;
        g.ldc = N;
        if (hw) { g.stats = &st; g.stats_hw = hw; }
        puts(gemm_kernel_name(g).c_str());
    }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    """rows of (M, N, K, rows per image of the output statistics or 0) -> kernel names"""
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(DRIVER)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950", "--offload-host-only", "-x", "hip",
                    str(d / "plan.cpp"), "-I" + os.path.join(PKG, "csrc"), "-L" + PKG, "-lsdu", "-Wl,-rpath," + PKG,
                    "-o", str(d / "plan")], check=True)

    def ask(rows):
        text = "".join("%d %d %d %d\n" % r for r in rows)
        return subprocess.run([str(d / "plan")], input=text, capture_output=True, text=True, check=True).stdout.split()

    return ask


def test_statistics_tiles_reach_two_images(plan):
    """With output statistics no tile may hold rows of a third image: the epilogues keep two."""
    rows = [(B * hw, N, K, hw) for hw in (64, 128, 144, 192, 240, 255, 256, 1024)  # (gemm_stats_supported)
            for B in (1, 3, 16, 64) for N, K in ((320, 320), (1280, 1280), (1280, 6400))]
    names = plan(rows)
    for (M, N, K, hw), name in zip(rows, names, strict=True):
        mt = int(name.split("<")[1].split(",")[0])
        worst = max((min(M, m0 + mt) - 1) // hw - m0 // hw for m0 in range(0, M, mt))
        assert worst <= 1, (M, N, K, hw, name)
