"""Launch shapes chosen by te_autotune where one launch runs several dispatches
side by side: the dispatch keeps its shape there, and the step's words are the
oracle's whatever the shapes (at these sizes the timings of one step hardly
differ, so each pass of the tuner leaves another mix of them)."""
import numpy as np
import pytest

import runs
import te_host

pytestmark = pytest.mark.gpu

CASES = {
    "37x12x9_tke": dict(nx=37, ny=12, nz=9, tke=1, initial_tke=3, rayleigh=1, cache_moisture_turbulence=1),
    "70x21x16_species7": dict(nx=70, ny=21, nz=16, species=7),
    "65x18x11_open": dict(nx=65, ny=18, nz=11, open_x=1, tke=1, initial_tke=3, weno_momentum=1),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_tuned_shapes_reach_batched_dispatches(gpu, name):
    cfg = te_host.config(noise_sigma=0.2, dz=1000.0, **CASES[name])
    run = te_host.Run(cfg)
    run.init_state()
    ref = runs.OracleRun(cfg)
    names, _ = run.program()
    start = run.launches()
    together = np.zeros(len(names), bool)  # run by a launch that runs others too
    for i, n in enumerate(start[:, 0]):
        together[i: i + n] |= n > 1
    assert start[:, 0].sum() == len(names) and together.any()
    end = runs.arena_end(run)
    keep = runs.state_mask(run)
    seen = set()
    for _ in range(4):
        run.autotune(reps=1, force=True)
        now = run.launches()
        assert np.array_equal(now[:, 0], start[:, 0])
        for i in np.nonzero(together & (now[:, 1:] != start[:, 1:]).any(axis=1))[0]:
            seen.add((names[i], tuple(now[i, 1:].tolist())))
        run.step(2)  # (a captured graph)
        run.sync()
        ref.step(2)
        got, want = run.read(0, end), ref.M[:end].copy()
        got[~keep] = 0
        want[~keep] = 0
        assert np.array_equal(got, want), runs.first_difference(run, got, want)
    print(name, sorted(seen), flush=True)
    assert seen
    run.close()
