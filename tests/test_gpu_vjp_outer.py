"""The gathered flux transpose's sums on the two outer planes.

<F, lamF> pairs what the wall planes emit outwards with the state of the outer
planes, once for the whole grid.  That is seen where the outer planes hold a
field and the wall planes' adjoint of it is not zero: BZ free on the walls
(ibcon 1), with BX, BY and BZ random on planes 0 and npz+1 as well.  Grids of
one plane a chunk (the planner's choice below 257 tiles; asserted on the CPU in
test_vjp_plan.py), one and two z ranks, and chunks of two planes and of more,
against the per-cell kernel with global atomics (R3D_ADJ_VJP=atomic).

Both sum the same entries; as in test_gpu_vjp_edges.py their rounding differs
by some 1e-13 of the largest gradient, a term paired twice shows at its size.
"""
import os

import numpy as np
import pytest

from conftest import load_package

pkg = load_package()
pytestmark = pytest.mark.gpu

# a strong, diffusive field (the advective limit still sets dt)
MAG = ["--lmag", "1", "--rm", "5", "--beta", "0.2", "--ampb", "1", "--bfh", "2", "--bzp", "10",
       "--ibcon", "1", "--re", "20", "--pr", "1"]
# npx, npy, npz, npez
GRIDS = [(33, 13, 10, 1), (33, 13, 10, 2), (24, 12, 48, 2), (65, 25, 14, 1), (34, 26, 61, 1),
         (100, 40, 90, 3)]


@pytest.mark.parametrize("grid", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_outer_planes_are_paired_once(grid):
    npx, npy, npz, npez = grid
    args = ["--npx", str(npx), "--npy", str(npy), "--npz", str(npz), "--npey", "1", "--npez",
            str(npez), "--tp", "0"] + MAG
    run = pkg.Run(args)
    x0 = {n: a.copy() for n, a in run.state().items()}
    rng = np.random.default_rng(npx * 1000 + npz)
    for n, x in x0.items():
        field = n in ("bx", "by", "bz")
        inner = x[slice(None) if field else slice(1, -1), 1:-1, 1:-1]
        r = rng.uniform(-1, 1, inner.shape)
        inner[:] = inner * (1.0 + 0.01 * r) if n in ("ro", "tt") else inner + (0.5 if field else 0.02) * r
        if field:  # periodic ghosts, on the outer planes too
            x[:, 0], x[:, -1] = x[:, -2], x[:, 1]
            x[:, :, 0], x[:, :, -1] = x[:, :, -2], x[:, :, 1]
    print(f"[gpu] outer planes, {' '.join(args)}", flush=True)
    out = []
    for mode in ("atomic", "tiled"):
        os.environ["R3D_ADJ_VJP"] = mode
        try:
            adj = pkg.Adjoint(run.cfg(), run.metrics(), 2)
        finally:
            del os.environ["R3D_ADJ_VJP"]
        adj.set_initial(x0)
        assert np.isfinite(adj.forward(6))
        out.append(adj.backward())
        adj.close()
    (ga, rea, tha), (gt, ret, tht) = out
    worst = {n: float(np.abs(ga[n] - gt[n]).max() / np.abs(ga[n]).max()) for n in ga}
    worst["re"] = abs(rea - ret) / abs(rea)
    worst["theta"] = abs(tha - tht) / max(abs(tha), 1e-300)
    print(f"[gpu] {worst}", flush=True)
    assert all(v <= 1e-11 for v in worst.values()), worst
