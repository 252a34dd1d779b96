"""The GEMM planner's choices, on the CPU: a small driver linked with the library asks for the kernel and
workspace of one GEMM per line."""
import os
import subprocess

import pytest

import tile_cases
from conftest import PKG

DRIVER = r"""
#include "sdu_internal.h"
#include <cstdio>
using namespace sdu;
int main() {
    static double st;
    int conv, a[8];
    while (scanf("%d %d %d %d %d %d %d %d %d", &conv, a, a + 1, a + 2, a + 3, a + 4, a + 5, a + 6, a + 7) == 9) {
        GemmArgs g{};
        if (conv) {  // B H W Ci Co
            g.amode = A_CONV3;
            g.Bn = a[0]; g.Hin = g.Ho = a[1]; g.Win = g.Wo = a[2]; g.Cin = a[3]; g.N = a[4];
            g.stride = 1;
            g.M = g.Bn * g.Ho * g.Wo;
            g.K = g.K1 = 9 * g.Cin;
            g.ldc = g.N;
        } else {  // M N K K2 residual GEGLU fp32 stats_hw
            g.M = a[0]; g.N = a[1]; g.K = a[2];
            g.lda = g.K1 = a[2] - a[3];
            if (a[3]) { g.A2 = (const f16*)&st; g.lda2 = a[3]; }
            g.ldc = a[5] ? g.N / 2 : g.N;
            if (a[4]) { g.res = (const f16*)&st; g.ldr = g.ldc; }
            g.geglu = a[5];
            g.out_mode = a[6] ? OUT_F32 : OUT_F16;
            if (a[7]) { g.stats = &st; g.stats_hw = a[7]; }
        }
        printf("%s %zu\n", gemm_kernel_name(g).c_str(), gemm_workspace_bytes(g));
    }
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    """rows of (1, B, H, W, Ci, Co) or (0, M, N, K, K2, residual, GEGLU, fp32 output, rows per image of the
    output statistics or 0) -> [(kernel, workspace bytes)]"""
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(DRIVER)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    subprocess.run([hipcc, "-O1", "-std=c++17", "--offload-arch=gfx950", "--offload-host-only", "-x", "hip",
                    str(d / "plan.cpp"), "-I" + os.path.join(PKG, "csrc"), "-L" + PKG, "-lsdu", "-Wl,-rpath," + PKG,
                    "-o", str(d / "plan")], check=True)

    def ask(rows):
        text = "".join(" ".join(str(int(v)) for v in (*r, *[0] * (9 - len(r)))) + "\n" for r in rows)
        out = subprocess.run([str(d / "plan")], input=text, capture_output=True, text=True, check=True).stdout
        return [(n, int(b)) for n, b in (line.split() for line in out.splitlines())]

    return ask


@pytest.mark.parametrize("conv", [True, False])
def test_tile_cases_reach_their_kernels(plan, conv):
    """A refit of the planner that moves a size of tile_cases fails here, rather than leave the kernel it
    was there for untested."""
    rows = tile_cases.CONV if conv else tile_cases.DENSE_TILES
    got = plan([(1, *r[:5]) for r in rows] if conv else [(0, *r[:4], *r[5:8], 0) for r in rows])
    for r, (name, ws) in zip(rows, got, strict=True):
        if r[-1] is None:
            assert name.split("<")[0] == r[-2], (r, name)
        else:
            assert name == r[-2] and (ws > 0) == (r[-1] != "whole"), (r, name, ws)


def test_statistics_tiles_reach_two_images(plan):
    """With output statistics no tile may hold rows of a third image: the epilogues keep two."""
    rows = [(0, B * hw, N, K, 0, 0, 0, 0, hw) for hw in (64, 128, 144, 192, 240, 255, 256, 1024)  # (gemm_stats_supported)
            for B in (1, 3, 16, 64) for N, K in ((320, 320), (1280, 1280), (1280, 6400))]
    for (_, M, N, K, *_, hw), (name, _) in zip(rows, plan(rows), strict=True):
        mt = int(name.split("<")[1].split(",")[0])
        worst = max((min(M, m0 + mt) - 1) // hw - m0 // hw for m0 in range(0, M, mt))
        assert worst <= 1, (M, N, K, hw, name)
