"""Sides beyond 2^15 cells, word for word against the oracle: the substep's
halo cells at nx, nx + 3 and ny + 3 need more than 16 bits there."""
import numpy as np
import pytest

import runs
import te_host

pytestmark = pytest.mark.gpu

CASES = {
    "32770x4x4": dict(nx=32770, ny=4, nz=4),
    "4x32770x4": dict(nx=4, ny=32770, nz=4),
    "32769x5x4_open_y": dict(nx=32769, ny=5, nz=4, open_y=1),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_wide_grid_bit_exact(gpu, name):
    cfg = te_host.config(dz=5000.0, nsound=4, dt=3.0, noise_sigma=0.2, **CASES[name])
    print("wide grid", name, flush=True)
    ref = runs.OracleRun(cfg)
    run = te_host.Run(cfg)
    run.init_state()
    run.step(1)
    run.sync()
    ref.step(1)
    end = runs.arena_end(run)
    keep = runs.state_mask(run)
    got, want = run.read(0, end), ref.M[:end].copy()
    got[~keep] = 0
    want[~keep] = 0
    assert np.array_equal(got, want), runs.first_difference(run, got, want)
    run.close()
