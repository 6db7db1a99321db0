"""Merged launches of the open-boundary step (bc_open_xy, ...) against the
reference's dispatch list: on the CPU the two programs run in the oracle, on
the GPU the fused step is compared with the oracle word for word.  One open
axis next to a periodic one, both open, and sides of 4 cells (every cell
within reach of a halo); the operations are the same, so the bits are."""
import numpy as np
import pytest

import runs
import te_host

CASES = {
    "open_x": dict(nx=21, ny=18, nz=10, open_x=1, tke=1, initial_tke=3, dissipative_heating=1),
    "open_y": dict(nx=18, ny=21, nz=10, open_y=1, tke=1, initial_tke=3, species=7),
    "open_xy_mass": dict(nx=17, ny=13, nz=9, open_x=1, open_y=1, tke=1, initial_tke=3, mass_conservation=1, umove=7.0,
                         vmove=2.0),
    "open_x_dry": dict(nx=4, ny=5, nz=8, open_x=1, moist=0),
    "open_y_narrow": dict(nx=70, ny=4, nz=6, open_y=1, weno_momentum=1),
    "open_xy_deep": dict(nx=66, ny=9, nz=40, open_x=1, open_y=1, tke=1, initial_tke=3, rayleigh=1),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_fused_open_program_equals_reference_program(name):
    cfg = te_host.config(**CASES[name])
    a, b = runs.OracleRun(cfg), runs.OracleRun(cfg, fused=True)
    assert len(b.names) < len(a.names) and not {"bc_open_x", "bc_open_y"} & set(b.names)
    a.step(2)
    b.step(2)
    end = runs.arena_end(a.enc)
    keep = runs.state_mask(a.enc)
    wa, wb = a.M[:end].copy(), b.M[:end].copy()
    wa[~keep] = 0
    wb[~keep] = 0
    assert np.array_equal(wa, wb), runs.first_difference(a, wa, wb)


@pytest.mark.gpu
@pytest.mark.parametrize("name", sorted(CASES))
def test_fused_open_step_bit_exact(gpu, name):
    cfg = te_host.config(**CASES[name])
    print("open boundary step", name, flush=True)
    ref = runs.OracleRun(cfg)
    run = te_host.Run(cfg)
    run.init_state()
    run.step(3)
    run.sync()
    ref.step(3)
    end = runs.arena_end(run)
    keep = runs.state_mask(run)
    got, want = run.read(0, end), ref.M[:end].copy()
    got[~keep] = 0
    want[~keep] = 0
    assert np.array_equal(got, want), runs.first_difference(run, got, want)
    run.close()
