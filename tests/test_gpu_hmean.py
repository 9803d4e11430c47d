"""The horizontal-mean chains at the sizes where their kernel can go wrong.

The chains of k_hmean_partial run through 192-value segments, in blocks of
4 or 8 chains, or alone through 704-value ones (at most 256 chains): rows shorter and longer than a segment, lengths just below,
at and just above whole segments, one chain a block (few planes), more chains
than fit four to a CU with a short last block, and one to six y ranks.  Each
sum runs in the reference's order, so the runs equal the oracle bit for bit.
"""
import sys

import numpy as np
import pytest

import oracle
from conftest import load_package

pkg = load_package()
pytestmark = pytest.mark.gpu

DEN = ["--ngrid", "0", "--id", "1", "--dh", "0.4", "--dv", "0.3"]
RLX = ["--ngrid", "0", "--itcon", "0", "--izcon", "1", "--rlax", "0.5", "--toff", "0.5",
       "--tstart", "-1"]
# npx, npy, npz, npey, npez
GRIDS = [
    (176, 4, 24, 1, 2),    # alone: exactly one segment a chain
    (703, 3, 24, 1, 2),    # rows one short of a segment
    (705, 4, 24, 2, 2),    # rows one over it
    (5, 7, 12, 1, 2),      # a chain shorter than a segment
    (192, 4, 128, 2, 2),   # 260 chains, four a block: rows of one segment
    (191, 6, 90, 3, 2),    # one short of it
    (193, 6, 90, 3, 2),    # one over it
    (64, 9, 128, 3, 2),    # exactly one segment a chain
    (400, 12, 174, 2, 3),  # rows of two segments and a bit
    (37, 30, 96, 6, 4),    # 588 chains: four a block
    (20, 18, 402, 3, 3),   # 1212 chains: eight a block, the last one short
]


@pytest.mark.parametrize("physics", ["density", "relax"])
@pytest.mark.parametrize("grid", GRIDS, ids=["x".join(map(str, g)) for g in GRIDS])
def test_chains_match_oracle(grid, physics):
    args = [a for f, v in zip(("--npx", "--npy", "--npz", "--npey", "--npez"), grid)
            for a in (f, str(v))] + (DEN if physics == "density" else RLX)
    print(f"[gpu] {physics} {grid}", flush=True)
    sys.stdout.flush()
    run = pkg.Run(args)
    sim = run.make_sim()
    orc = oracle.Sim(args)
    sim.step(2)
    orc.step(2)
    for r in range(orc.nranks):
        for n, a in sim.download_rank(r, ["ru", "rv", "rw", "ro", "tt"]).items():
            assert np.array_equal(a.view(np.uint64), orc.field(r, n).view(np.uint64)), (r, n)
    so, sg = orc.scalars(), sim.scalars()
    assert so["dt"] == sg["dt"] and so["timc"] == sg["timc"]
    sim.close()
