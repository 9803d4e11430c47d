"""The adjoint of the time step: its least limit found among listed cells.

The gathered transpose lists the cells that may hold a step's least limit, and
k_dt_adj takes the exact limits of those; with none or more than 1024 of them
it goes over the whole state.  With the scattered transpose
(R3D_ADJ_VJP=atomic) nothing is listed, so every step goes over the state:
both have to find the same cell.  Noisy states (a few cells listed) and states
uniform in x and y, where every cell of a plane has the same limits: 900, 1024
and 1200 listed, ties going to the first cell.

The two transposes sum the same entries and differ by their rounding, 1e-13 of
the largest gradient over the three steps, and another cell's limits would show
at their full size: 1e-11, as for the other comparisons of the two kernels.
"""
import os

import numpy as np
import pytest

from conftest import load_package

pkg = load_package()
pytestmark = pytest.mark.gpu

MAG = ["--lmag", "1", "--rm", "50", "--beta", "10", "--ampb", "1", "--bfh", "2", "--bzp", "10"]
# npx, npy, npz, uniform, fixed dt, extra flags
CASES = [(33, 13, 20, False, 0.0, []), (33, 13, 20, False, 0.0, MAG), (33, 13, 20, False, 1e-3, []),
         (30, 30, 20, True, 0.0, []), (32, 32, 20, True, 0.0, []), (40, 30, 20, True, 0.0, []),
         (30, 30, 20, True, 0.0, MAG), (40, 30, 20, True, 0.0, MAG)]


@pytest.mark.parametrize("case", CASES, ids=[f"{n}" for n in range(len(CASES))])
def test_listed_limit_equals_full_pass(case):
    npx, npy, npz, uniform, fixed, extra = case
    args = ["--npx", str(npx), "--npy", str(npy), "--npz", str(npz), "--npey", "1", "--npez", "1",
            "--tp", "0"] + extra
    run = pkg.Run(args)
    x0 = {n: a.copy() for n, a in run.state().items()}
    rng = np.random.default_rng(npx)
    inner = (slice(1, -1),) * 3
    for n in x0:
        x = x0[n][inner]
        if uniform:
            x[:] = x.mean(axis=(1, 2), keepdims=True)
        shape = (x.shape[0], 1, 1) if uniform else x.shape
        r = rng.uniform(-1, 1, shape)
        x[:] = x * (1.0 + 0.01 * r) if n in ("ro", "tt") else x + 0.02 * r
    print(f"[gpu] dt adjoint, {case}", flush=True)
    out = []
    for mode in ("atomic", "tiled"):
        os.environ["R3D_ADJ_VJP"] = mode
        try:
            adj = pkg.Adjoint(run.cfg(), run.metrics(), 2)
        finally:
            del os.environ["R3D_ADJ_VJP"]
        if fixed:
            adj.set_fixed_dt(fixed)
        adj.set_initial(x0)
        assert np.isfinite(adj.forward(3))
        out.append(adj.backward())
        again = adj.backward()  # the lists start empty again
        for n in again[0]:
            assert np.abs(again[0][n] - out[-1][0][n]).max() <= 1e-11 * np.abs(again[0][n]).max(), n
        adj.close()
    (ga, rea, tha), (gt, ret, tht) = out
    for n in ga:
        scale = np.abs(ga[n]).max()
        assert np.isfinite(scale) and np.abs(ga[n] - gt[n]).max() <= 1e-11 * scale, n
    assert abs(rea - ret) <= 1e-11 * abs(rea)
