"""The gathered flux transpose at the sizes where it can go wrong.

k_vjp collects every cell's entries from its neighbours over 32 x 12 tiles and
z chunks, with one-sided stencils that reach two and three planes in from the
walls.  Here against the per-cell kernel with global atomics
(R3D_ADJ_VJP=atomic), on random states: the smallest grid (every plane near
both walls, x and y narrower than the tile's halo), one below, at and above
the tile in x and y, two tiles and one more cell, a chunk boundary at each of
the planes the walls reach, one and two z ranks (the bottom wall's one-sided
field stencils are off with one), both bottom conditions, BZ free on the
walls, rotation.

Both sum the same entries, some 150 products per cell of which the largest
set the scale, over three steps of three stages: their rounding differs by a
few hundred units of 1e-16 at most, 1e-13; 1e-11 as for the other
comparisons of the two kernels.
"""
import os

import numpy as np
import pytest

from conftest import load_package

pkg = load_package()
pytestmark = pytest.mark.gpu

MAG = ["--lmag", "1", "--rm", "50", "--beta", "10", "--ampb", "1", "--bfh", "2", "--bzp", "10"]
ROT = ["--lrot", "1", "--ry", "0.2", "--ang", "0.3"]
# npx, npy, npz, npey, npez, extra flags
GRIDS = [
    (3, 3, 6, 1, 1, []), (3, 3, 6, 1, 2, MAG), (4, 5, 7, 1, 1, MAG),
    (31, 11, 8, 1, 2, ROT), (32, 12, 9, 1, 3, MAG + ROT), (33, 13, 10, 1, 2, MAG),
    (64, 24, 12, 2, 2, ["--izcon", "1"]), (65, 25, 14, 1, 1, MAG + ["--izcon", "1"]),
    (20, 14, 260, 1, 2, []), (34, 26, 61, 1, 1, MAG + ["--ibcon", "1"]),
    (100, 7, 33, 1, 3, MAG + ["--itcon", "0"]),
]


@pytest.mark.parametrize("grid", GRIDS, ids=["x".join(map(str, g[:3])) + f"_{n}"
                                             for n, g in enumerate(GRIDS)])
def test_gathered_transpose_equals_scattered(grid):
    npx, npy, npz, npey, npez, extra = grid
    # the host set-up's profile needs nine planes: a lower grid is its top part
    nz = max(npz, 9)
    args = ["--npx", str(npx), "--npy", str(npy), "--npz", str(nz), "--npey", str(npey),
            "--npez", str(npez if nz == npz else 1), "--tp", "0"] + extra
    run = pkg.Run(args)
    x0 = {n: a[:npz + 2].copy() for n, a in run.state().items()}
    cfg, met = run.cfg(), run.metrics()
    cfg.npz, cfg.npez = npz, npez
    for n in pkg.METRIC_NAMES[8:]:
        met[n] = met[n][:npz + 2].copy()
    rng = np.random.default_rng(npx * 1000 + npz)
    inner = (slice(1, -1),) * 3
    for n in x0:
        r = rng.uniform(-1, 1, x0[n][inner].shape)
        if n in ("ro", "tt"):
            x0[n][inner] *= 1.0 + 0.01 * r
        else:
            x0[n][inner] += 0.02 * r
    print(f"[gpu] gathered vs scattered transpose, {npx}x{npy}x{npz} {' '.join(args[6:])}", flush=True)
    out = []
    for mode in ("atomic", "tiled"):
        os.environ["R3D_ADJ_VJP"] = mode
        try:
            adj = pkg.Adjoint(cfg, met, 2)
        finally:
            del os.environ["R3D_ADJ_VJP"]
        adj.set_initial(x0)
        J = adj.forward(3)
        assert np.isfinite(J)
        out.append(adj.backward())
        adj.close()
    (ga, rea, tha), (gt, ret, tht) = out
    for n in ga:
        scale = np.abs(ga[n]).max()
        assert np.isfinite(scale) and np.abs(ga[n] - gt[n]).max() <= 1e-11 * scale, n
        ghost = gt[n].copy()
        ghost[inner] = 0.0
        assert not ghost.any(), f"{n}: ghost entries"
    assert abs(rea - ret) <= 1e-11 * abs(rea) and abs(tha - tht) <= 1e-11 * max(abs(tha), 1e-300)
