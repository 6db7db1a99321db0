"""Merged launches around the scalars' advection against the reference's
dispatch list in the oracle, word for word (halo cells included): the sizes
where a cell is the source of several halo cells (sides of 4 to 7) or a row
ends in a partly filled wave, every boundary kind, the flux kinds, and fields
that go negative so that the positive-definite correction acts.  The
arithmetic is the reference's, operation by operation, so the bits are equal."""
import numpy as np
import pytest

import runs
import te_host

pytestmark = pytest.mark.gpu

CASES = {
    "4x4x4": dict(nx=4, ny=4, nz=4),
    "5x7x6_open_x": dict(nx=5, ny=7, nz=6, open_x=1, tke=1, initial_tke=3),
    "7x4x5_open_y": dict(nx=7, ny=4, nz=5, open_y=1, species=7),
    "65x6x9_open": dict(nx=65, ny=6, nz=9, open_x=1, open_y=1, tke=1, initial_tke=3, cache_moisture_turbulence=1),
    "130x5x12_flx5": dict(nx=130, ny=5, nz=12, weno_scalars=0, tke=1, initial_tke=3, cache_moisture_turbulence=0),
    "63x9x17": dict(nx=63, ny=9, nz=17, species=7, tke=1, initial_tke=3, cache_moisture_turbulence=1, rayleigh=1),
    "64x5x40_weno": dict(nx=64, ny=5, nz=40, weno_momentum=1, species=11),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_merged_scalar_launches_bit_exact(gpu, name):
    cfg = te_host.config(noise_sigma=0.2, **CASES[name])
    print("merged scalar launches", name, flush=True)
    ref = runs.OracleRun(cfg)
    run = te_host.Run(cfg)
    run.init_state()
    rng = np.random.default_rng(len(name))
    n = run.sJ * run.sK * (run.nz + 1)
    scalars = [f for f in run.fields if f + "_a" in run.fields and f.startswith("q")]
    assert scalars
    for f in scalars:  # sparse spikes next to zeros, and other words in every halo cell
        q = np.where(rng.random(n) < 0.2, rng.random(n) * 4e-3, 0.0).astype(np.float32)
        for s in (f, f + "_a"):
            run.upload(run.field_offset(s), q.view(np.uint32))
            o = ref.enc.field_offset(s)
            ref.M[o: o + n] = q.view(np.uint32)
    for _ in range(2):
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
