"""The stage kernel's split into tiles and z chunks (r3d_plan.hpp), on the CPU.

Over a wide range of grids the planned chunks cover every plane once, have at
least the three planes the walls' extrapolation reads and fit the 128 planes
of z metrics a tile stages, the small tile is taken only where every tile has a
CU (and not by the contracted variant, which is built without it), no split has more than 32 times
as many tiles as CUs unless the grid needs them at 128-plane chunks, forced
tilings are taken as given, and r3d_hip_step_noalloc's static scratch (131072
doubles, five per tile and boundary block) accepts exactly the grids it
accepted when chunks were the largest of 128..8 planes giving 2048 tiles.
"""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include <cstdlib>
#include "r3d_plan.hpp"
using namespace r3d;
static bool covers(const StagePlan& p, int npz) {
    int next = 1;
    for (int kz = 0; kz < p.nkc; ++kz) {  // as the kernel forms k0 and k1
        const int k0 = 1 + p.kq * kz + (kz < p.krem ? kz : p.krem);
        int k1 = k0 + p.kq - 1 + (kz < p.krem ? 1 : 0);
        if (k1 > npz) k1 = npz;
        if (k0 != next || k1 < k0 || k1 - k0 + 1 > KC_MAX || k1 - k0 + 1 < KC_MIN || k1 - k0 + 1 > p.kc) return false;
        next = k1 + 1;
    }
    return next == npz + 1;
}
int main(int argc, char** argv) {
    const bool lmag = atoi(argv[1]), feature = atoi(argv[2]);
    long bad = 0, n = 0;
    for (int x = 3; x <= 2600; x = x * 4 / 3 + 1)
        for (int y = 3; y <= 2600; y = y * 5 / 4 + 1)
            for (int z = 6; z <= 6000; z = z * 9 / 8 + 1, ++n) {
                const StagePlan p = plan_stage(x, y, z, lmag, feature, false, 0, 0, 256);
                StagePlan o = stage_tiles(x, y, lmag, lmag ? TILE_Y_MAG : feature ? 8 : hydro_tile_rows(y));
                for (int kc : {128, 64, 32, 16, 8}) {
                    chunks_of(o, z, kc);
                    if (o.blocks() >= 2048) break;
                }
                const long nbb = ((x + 2L) * (y + 2) + 255) / 256;
                const bool was = (o.blocks() + 2 * nbb) * 5 <= 131072;
                const bool is = (p.blocks() + 2 * nbb) * 5 <= 131072;
                const bool ok = covers(p, z) && was == is && stage_cost(p, 256) <= stage_cost(o, 256) &&
                                (p.blocks() <= 32 * 256 || p.blocks() == o.blocks()) &&
                                (!feature || lmag || p.ty == 8) &&
                                (p.tw != TILE_W_SMALL || p.blocks() <= 256) &&
                                plan_stage(x, y, z, lmag, feature, true, 0, 0, 256).tw != TILE_W_SMALL;
                if (!ok && bad++ < 5) printf("%d x %d x %d: ty %d kc %d nkc %d\n", x, y, z, p.ty, p.kc, p.nkc);
                for (int kc : {8, 128}) {
                    const StagePlan f = plan_stage(x, y, z, lmag, feature, false, o.ty, kc, 256);
                    if (!covers(f, z) || f.kc != kc || f.ty != o.ty) ++bad;
                }
            }
    printf("%ld grids, %ld bad\n", n, bad);
    return bad != 0;
}
"""


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src = d / "plan.cpp"
    src.write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "rast-3dmhd_amd", "csrc"),
                    "-o", str(d / "plan"), str(src)], check=True)
    return str(d / "plan")


@pytest.mark.parametrize("lmag,feature", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_planned_chunks_cover_the_grid(exe, lmag, feature):
    r = subprocess.run([exe, str(lmag), str(feature)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
