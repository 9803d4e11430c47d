"""The flux transpose's split into tiles and z chunks (plan_vjp), on the CPU.

Over a wide range of grids and CU counts the chunks cover every plane once, have
at least one plane and at most the VJP_KC planes of metrics that a tile stages,
and exactly one chunk starts at plane 1 and one ends at plane npz (those pair
the outer planes' sums); the grids of test_gpu_vjp_outer.py have the chunk sizes
that it names.
"""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = r"""
#include <cstdio>
#include "r3d_plan.hpp"
using namespace r3d;
int main() {
    long n = 0, bad = 0;
    for (int cus : {1, 32, 256, 304})
        for (int x = 3; x <= 2600; x = x * 4 / 3 + 1)
            for (int y = 3; y <= 2600; y = y * 5 / 4 + 1)
                for (int z = 6; z <= 6000; z = z * 9 / 8 + 1, ++n) {
                    const VjpPlan p = plan_vjp(x, y, z, cus);
                    int next = 1, first = 0, last = 0;
                    bool ok = p.ntx * VW >= x && p.nty * VH >= y;
                    for (int kz = 0; kz < p.nkc; ++kz) {  // as the kernel forms k0 and k1
                        const int k0 = 1 + p.kq * kz + (kz < p.krem ? kz : p.krem);
                        const int k1 = k0 + p.kq - 1 + (kz < p.krem ? 1 : 0);
                        ok = ok && k0 == next && k1 >= k0 && k1 - k0 < VJP_KC;
                        first += k0 == 1;
                        last += k1 == z;
                        next = k1 + 1;
                    }
                    if ((!ok || next != z + 1 || first != 1 || last != 1) && bad++ < 5)
                        printf("%d x %d x %d, %d CUs: nkc %d kq %d krem %d\n", x, y, z, cus, p.nkc,
                               p.kq, p.krem);
                }
    for (auto& g : {VjpPlan{33, 13, 10, 1, 0}, VjpPlan{24, 12, 48, 1, 0}, VjpPlan{65, 25, 14, 1, 0},
                    VjpPlan{34, 26, 61, 1, 30}})  // npx, npy, npz, then kq and krem on 256 CUs
        if (const VjpPlan p = plan_vjp(g.ntx, g.nty, g.nkc, 256); p.kq != g.kq || p.krem != g.krem) {
            printf("%d x %d x %d: kq %d krem %d\n", g.ntx, g.nty, g.nkc, p.kq, p.krem);
            ++bad;
        }
    printf("%ld grids, %ld bad\n", n, bad);
    return bad != 0;
}
"""


def test_planned_chunks_cover_the_grid(tmp_path):
    (tmp_path / "plan.cpp").write_text(SRC)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I" + os.path.join(ROOT, "rast-3dmhd_amd", "csrc"),
                    "-o", str(tmp_path / "plan"), str(tmp_path / "plan.cpp")], check=True)
    r = subprocess.run([str(tmp_path / "plan")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
