"""Radiation boundary speeds and the mass sums, which add in a fixed order from
tiles formed side by side, against the oracle word for word: rows and levels on
either side of the tile sizes (16 rows, 64 columns, 64 levels)."""
import numpy as np
import pytest

import runs
import te_host

pytestmark = pytest.mark.gpu

GRIDS = [(5, 4, 4), (16, 17, 5), (63, 15, 8), (65, 33, 64), (64, 16, 65), (130, 9, 70)]


@pytest.mark.parametrize("fuse", [0, 1])
@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "%dx%dx%d" % g)
def test_open_edges_and_mass_sums_bit_exact(gpu, grid, fuse):
    nx, ny, nz = grid
    cfg = te_host.config(nx=nx, ny=ny, nz=nz, dz=20000.0 / nz, nsound=4, dt=3.0, noise_sigma=0.2, open_x=1, open_y=1,
                         mass_conservation=1, umove=5.0, vmove=-3.0, fuse=fuse)
    print("open edges", grid, fuse, flush=True)
    ref = runs.OracleRun(cfg)
    run = te_host.Run(cfg)
    run.init_state()
    run.step(2)
    run.sync()
    ref.step(2)
    end = runs.arena_end(run)
    keep = runs.state_mask(run)
    got, want = run.read(0, end), ref.M[:end].copy()
    got[~keep] = 0
    want[~keep] = 0
    assert np.array_equal(got, want), runs.first_difference(run, got, want)
    run.close()
