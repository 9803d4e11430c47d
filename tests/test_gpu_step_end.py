"""The end of a step, at the border between its one-launch and two-launch forms.

768 stage tiles and fewer reduce the time-step partials and, where the screen
could not prove them, redo the limits exactly in one launch; more take two.
Either way every step's dt and umach are the oracle's, with the default margin
of the screen, one that always takes the exact pass and one that evaluates
every cell.
"""
import numpy as np
import pytest

import oracle
from conftest import load_package

pkg = load_package()
pytestmark = pytest.mark.gpu

MAG = ["--lmag", "1", "--rm", "50", "--beta", "10", "--ampb", "1", "--bfh", "2", "--bzp", "10"]
# npx, npy, npz, tile rows, the tiles expected, extra flags
CASES = [(12, 4, 16, 0, 2, []), (192, 64, 256, 8, 768, []), (192, 64, 264, 8, 792, []),
         (96, 96, 256, 0, 768, MAG), (96, 96, 264, 0, 792, MAG)]


@pytest.mark.parametrize("margin", [0.0, -0.5, 1e9])
@pytest.mark.parametrize("case", CASES, ids=[f"{c[4]}tiles{'_mhd' if c[5] else ''}" for c in CASES])
def test_step_end_matches_oracle(case, margin):
    npx, npy, npz, rows, tiles, extra = case
    args = ["--npx", str(npx), "--npy", str(npy), "--npz", str(npz), "--npey", "1", "--npez",
            "2"] + extra
    print(f"[gpu] {' '.join(args)} margin={margin}", flush=True)
    run = pkg.Run(args)
    sim = run.make_sim(tile_rows=rows, zchunk=8, dt_screen=margin)
    assert np.prod(sim.tiling()[2:5]) == tiles, sim.tiling()
    orc = oracle.Sim(args)
    for _ in range(3):
        sim.step(1)
        orc.step(1)
        so, sg = orc.scalars(), sim.scalars()
        for k in ("dt", "timc", "umach", "nit"):
            assert so[k] == sg[k], k
    sim.close()
