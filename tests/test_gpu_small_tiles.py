"""Stage tiles at the edges of their ranges, against the oracle bit for bit.

The 4 x 16 tile of small hydro grids (rows and columns one below, at and one
above the tile, the smallest grid); chunks of three planes with one more in
the first ones; a forced chunk whose last one would have fewer than the three
planes that the walls' extrapolation reads (33 planes: equal chunks are taken);
one chunk with both walls; each wall condition, in full and truncated steps,
every field with its ghost cells, the outer planes among them.
"""
import numpy as np
import pytest

import oracle
from conftest import load_package

pkg = load_package()
pytestmark = pytest.mark.gpu

X = ["ru", "rv", "rw", "ro", "tt"]
MAG = ["--lmag", "1", "--rm", "50", "--beta", "10", "--ampb", "1", "--bfh", "2", "--bzp", "10"]
# npx, npy, npz, npey, npez, zchunk, the tile rows expected, extra flags
CASES = [
    (16, 16, 32, 2, 2, 0, 4, []), (15, 3, 9, 1, 1, 0, 4, ["--tp", "0"]),
    (17, 5, 10, 1, 2, 0, 4, ["--izcon", "1"]), (3, 4, 9, 1, 1, 0, 4, ["--itcon", "0"]),
    (33, 13, 31, 1, 1, 0, 4, ["--itcon", "4"]), (48, 20, 50, 2, 2, 0, 4, ["--tp", "0"]),
    (64, 64, 50, 2, 2, 0, 8, []), (70, 18, 33, 2, 3, 8, 9, []), (70, 18, 33, 2, 3, 16, 9, []),
    (40, 17, 33, 1, 3, 32, 9, ["--itcon", "0", "--tp", "0"]),
    (70, 25, 33, 5, 3, 8, 12, MAG), (33, 13, 11, 1, 1, 0, 12, MAG + ["--ibcon", "1"]),
]


@pytest.mark.parametrize("nstages", [3, 2, 1])
@pytest.mark.parametrize("case", CASES, ids=["x".join(map(str, c[:3])) + f"_kc{c[5]}"
                                             for c in CASES])
def test_small_tiles_and_short_chunks_match_oracle(case, nstages):
    npx, npy, npz, npey, npez, zchunk, rows, extra = case
    args = ["--npx", str(npx), "--npy", str(npy), "--npz", str(npz), "--npey", str(npey),
            "--npez", str(npez)] + extra
    print(f"[gpu] {' '.join(args)} zchunk={zchunk} stages={nstages}", flush=True)
    run = pkg.Run(args)
    sim = run.make_sim(zchunk=zchunk)
    assert sim.tiling()[0] == rows, sim.tiling()
    orc = oracle.Sim(args)
    sim.step(2)
    orc.step(2)
    sim.step(1, nstages)
    orc.step(1, nstages)
    names = X + (["bx", "by", "bz"] if "--lmag" in args else [])
    for r in range(orc.nranks):
        got = sim.download_rank(r, names + ["z" + n for n in names])
        for n, g in got.items():
            w = orc.field(r, n)
            if n.startswith("z"):
                g, w = g[1:-1, 1:-1, 1:-1], w[1:-1, 1:-1, 1:-1]
            assert np.array_equal(g.view(np.uint64), w.view(np.uint64)), (r, n)
    so, sg = orc.scalars(), sim.scalars()
    for k in ("dt", "timc", "umach", "nit"):
        assert so[k] == sg[k], k
    sim.close()
