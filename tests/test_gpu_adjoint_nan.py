"""The gradient of a run that blew up.

Where every cell's limits are no numbers (a density of NaN), no cell sets dt:
k_dt_adj finds no least limit, among its listed cells (640 of them) or over the
whole state (8580), and adds nothing.  J and the gradients are NaN then, as plain
arithmetic gives them, on both transposes.  With LMAG the resistive limit is
still a number and some cell keeps setting dt.
"""
import os

import numpy as np
import pytest

from conftest import load_package

pkg = load_package()
pytestmark = pytest.mark.gpu

MAG = ["--lmag", "1", "--rm", "50", "--beta", "10", "--ampb", "1", "--bfh", "2", "--bzp", "10"]


@pytest.mark.parametrize("extra", [[], MAG], ids=["hydro", "mhd"])
@pytest.mark.parametrize("mode", ["tiled", "atomic"])
@pytest.mark.parametrize("grid", [(8, 8, 10), (33, 13, 20)], ids=["listed", "whole"])
def test_nan_state_has_a_nan_gradient(grid, mode, extra):
    npx, npy, npz = grid
    args = ["--npx", str(npx), "--npy", str(npy), "--npz", str(npz), "--npey", "1", "--npez", "1",
            "--tp", "0"] + extra
    print(f"[gpu] gradient of a NaN state, {' '.join(args)} {mode}", flush=True)
    run = pkg.Run(args)
    x0 = run.state()
    x0["ro"][:] = np.nan
    os.environ["R3D_ADJ_VJP"] = mode
    try:
        adj = pkg.Adjoint(run.cfg(), run.metrics(), 2)
    finally:
        del os.environ["R3D_ADJ_VJP"]
    adj.set_initial(x0)
    assert np.isnan(adj.forward(3))
    grad, _, _ = adj.backward()
    assert np.isnan(grad["ru"][1:-1, 1:-1, 1:-1]).all()
    # the context is good for the next run
    adj.set_initial(run.state())
    assert np.isfinite(adj.forward(3))
    grad, re, th = adj.backward()
    assert all(np.isfinite(grad[n]).all() for n in grad) and np.isfinite(re) and np.isfinite(th)
    adj.close()
