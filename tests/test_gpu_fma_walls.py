"""Rounding where the FMA-contracted builds must not contract.

Variant 1 contracts the fluxes, not the wall cells: the boundary conditions, and
the wall cells' time-step limits and Mach number, round every product and sum by
themselves, as the exact pass over a state does.  The state is driven so that
the wall cells set both extrema; expected values are numpy's from the downloaded
state, bit for bit.

The adjoint (contracted too) takes the cell that sets dt from limits that round
like the forward's: on states that are uniform but for a few units in the last
place the gradient with the time step's own derivative and the one without
differ at exactly the cell where numpy's limits have their first minimum.
"""
import numpy as np
import pytest

from conftest import load_package

pkg = load_package()
pytestmark = pytest.mark.gpu

MAG = ["--lmag", "1", "--rm", "50", "--beta", "10", "--ampb", "1", "--bfh", "2", "--bzp", "10"]


def limits(c, met, x):
    """ogamma*UU/T and the time-step limits (list) per cell, ghosts cut off, in
    the order of operations of the reference (src/step.cpp:125-209)."""
    inner = {n: a[1:-1, 1:-1, 1:-1] for n, a in x.items()}
    ru, rv, rw, ro, tt = (inner[n] for n in ("ru", "rv", "rw", "ro", "tt"))
    dd = np.minimum(np.minimum(met["ddx"][1:-1][None, None, :], met["ddy"][1:-1][None, :, None]),
                    met["ddz"][1:-1][:, None, None])
    uu = (ru * ru + rv * rv + rw * rw) * (1.0 / ro) * (1.0 / ro)
    um = (1.0 / c.gamma) * uu / tt
    if c.lmag:
        bx, by, bz = (inner[n] for n in ("bx", "by", "bz"))
        b2 = (bx * bx + by * by + bz * bz) * c.obeta / ro
        fast = uu + c.gamma * tt + b2 + 2.0 * np.sqrt(uu * (c.gamma * tt + b2))
    else:
        fast = uu + c.gamma * tt + 2.0 * np.sqrt(uu * c.gamma * tt)
    out = [dd / np.sqrt(fast), 0.5 * dd * dd * c.repr * c.cv * ro / met["rkapa"][1:-1][:, None, None],
           0.375 * dd * dd * c.re * ro]
    if c.lmag:
        out.append(0.5 * dd * dd * c.rm + 0.0 * ro)
    return um, out


@pytest.mark.parametrize("seed", range(4))
@pytest.mark.parametrize("extra", [[], MAG], ids=["hydro", "mhd"])
def test_wall_cells_of_the_fma_variant_round_exactly(extra, seed):
    # flux conditions on both walls: T is extrapolated there
    args = ["--npx", "24", "--npy", "16", "--npz", "32", "--npey", "1", "--npez", "2", "--tp", "0",
            "--izcon", "1", "--ngrid", "0", "--re", "200", "--pr", "1"] + extra
    print(f"[gpu] FMA walls, seed {seed}: {' '.join(args)}", flush=True)
    run = pkg.Run(args)
    met, x = run.metrics(), {n: a.copy() for n, a in run.state().items()}
    rng = np.random.default_rng(seed)
    for n in ("ru", "rv"):
        # strong on the planes next to the walls, weak beyond them: BCON extrapolates
        # the largest speeds onto the walls
        for k in (2, -3):
            x[n][k, 1:-1, 1:-1] = x["ro"][k, 1:-1, 1:-1] * (3.0 + 0.1 * rng.uniform(-1, 1, x[n][k, 1:-1, 1:-1].shape))
    cfg = run.cfg()
    cfg.variant = 1
    sim = pkg.HipSim(cfg)
    sim.set_metrics(met)
    sim.upload_global(x)
    sim.set_scalars()
    for _ in range(3):
        sim.step(1)
        got = sim.download_global(list(x))
        c23dz = [cfg.c23 * (cfg.dzf / met["dzzdz"][k]) for k in (1, cfg.npz)]
        for k, d, flux in ((1, 1, -(c23dz[0] * cfg.theta)),
                           (cfg.npz, -1, c23dz[1] * cfg.theta / met["rkapa"][cfg.npz])):
            at = (slice(1, -1), slice(1, -1))
            t1, t2 = got["tt"][k + d][at], got["tt"][k + 2 * d][at]
            want = cfg.c43 * t1 - cfg.c13 * t2 + flux
            assert np.array_equal(got["tt"][k][at], want), f"tt on plane {k}"
            for n in ("ru", "rv"):
                q = got["ro"][k][at] * (cfg.c43 * got[n][k + d][at] / got["ro"][k + d][at] -
                                        cfg.c13 * got[n][k + 2 * d][at] / got["ro"][k + 2 * d][at])
                assert np.array_equal(got[n][k][at], q), f"{n} on plane {k}"
        um, lim = limits(cfg, met, got)
        wall = lambda a: a[[0, -1]]
        least = np.minimum.reduce([q.min() for q in lim])
        assert um.argmax() // um[0].size in (0, cfg.npz - 1) and wall(lim[0]).min() == least
        sim.step(1)  # takes the dt and umach that the step before reduced
        sc = sim.scalars()
        assert sc["dt"] == cfg.sff * least and sc["umach"] == np.sqrt(um.max())
    sim.close()


@pytest.mark.parametrize("seed", range(4))
@pytest.mark.parametrize("grid", [(12, 10, 8), (33, 13, 20)], ids=["listed", "whole"])
def test_dt_cell_rounds_like_the_forward(grid, seed):
    npx, npy, npz = grid
    nz = max(npz, 9)
    args = ["--npx", str(npx), "--npy", str(npy), "--npz", str(nz), "--npey", "1", "--npez", "1",
            "--tp", "0", "--ngrid", "0", "--re", "2000", "--pr", "1", "--xmax", "20", "--ymax", "20"]
    print(f"[gpu] dt cell, seed {seed}: {' '.join(args)}", flush=True)
    run = pkg.Run(args)
    met, x = run.metrics(), {n: a[:npz + 2].copy() for n, a in run.state().items()}
    cfg = run.cfg()
    cfg.npz = npz
    for n in pkg.METRIC_NAMES[8:]:
        met[n] = met[n][:npz + 2].copy()
    rng = np.random.default_rng(seed)
    base = {"ru": 0.37, "rv": -0.21, "rw": 0.13, "ro": 1.3, "tt": 1.7}
    for n, v in base.items():
        x[n][:] = v * (1.0 + 2.0 ** -52 * rng.integers(0, 4, x[n].shape))
    _, lim = limits(cfg, met, x)
    assert lim[0].min() < min(q.min() for q in lim[1:])  # the advective limit sets dt
    want = np.unravel_index(int(lim[0].argmin()), lim[0].shape)
    adj = pkg.Adjoint(cfg, met, 2)
    adj.set_initial(x)
    adj.forward(1)
    free, _, _ = adj.backward()
    adj.set_fixed_dt(cfg.sff * float(lim[0].min()))
    adj.forward(1)
    fixed, _, _ = adj.backward()
    adj.close()
    d = np.abs(free["tt"] - fixed["tt"])[1:-1, 1:-1, 1:-1]
    at = np.unravel_index(int(d.argmax()), d.shape)
    assert d.max() > 1e-6 * np.abs(fixed["tt"]).max() and at == want, (at, want, d.max())
    d[at] = 0.0
    assert d.max() <= 1e-12 * np.abs(fixed["tt"]).max(), d.max()
