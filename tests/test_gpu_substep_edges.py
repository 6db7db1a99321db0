"""One-launch acoustic substep (ac_column) and its neighbours at the sizes where
its split can go wrong, word for word against the oracle: levels dealt to 8
waves (fewer than 8, each remainder, both forms of the sweep's operands at 48 |
49 levels, the deepest 128), rows of a few columns up to a second and third
workgroup of one (64 | 65, 128 | 129, nx - 4 and nx - 1 in different ones),
sides short enough that a cell has two images per axis (4 to 6), and pivots
outside the range of the refined reciprocal.  The arithmetic is the
reference's, operation by operation, so the bits are equal."""
import numpy as np
import pytest

import runs
import te_host

pytestmark = pytest.mark.gpu

GRIDS = [(4, 4, 4), (5, 4, 7), (6, 6, 8), (7, 5, 9), (8, 7, 15), (12, 9, 17), (61, 7, 33), (64, 8, 40), (65, 6, 41),
         (66, 5, 48), (67, 7, 49), (68, 4, 56), (127, 5, 57), (129, 6, 64), (131, 4, 65), (33, 7, 80), (70, 8, 95),
         (20, 6, 97), (9, 8, 104), (66, 7, 121), (10, 5, 128)]


def compare(run, ref):
    end = runs.arena_end(run)
    keep = runs.state_mask(run)
    got, want = run.read(0, end), ref.M[:end].copy()
    got[~keep] = 0
    want[~keep] = 0
    assert np.array_equal(got, want), runs.first_difference(run, got, want)


@pytest.mark.parametrize("grid", GRIDS, ids=lambda g: "%dx%dx%d" % g)
def test_substep_split_bit_exact(gpu, grid):
    nx, ny, nz = grid
    cfg = te_host.config(nx=nx, ny=ny, nz=nz, dz=20000.0 / nz, nsound=4, dt=3.0, noise_sigma=0.2, kdiv=0.1)
    print("substep", grid, flush=True)
    ref = runs.OracleRun(cfg)
    run = te_host.Run(cfg)
    run.init_state()
    run.step(2)
    run.sync()
    ref.step(2)
    compare(run, ref)
    run.close()


@pytest.mark.parametrize("theta", [1e22, 1e26])
def test_substep_pivots_beyond_the_reciprocal_range(gpu, theta):
    """A potential temperature so large that the w row's pivots leave
    [2^-64, 2^64] in every column (1e26) or nearly (1e22): the first substep."""
    cfg = te_host.config(nx=70, ny=6, nz=20, dz=1000.0, nsound=4, noise_sigma=0.2)
    ref = runs.OracleRun(cfg, fused=True)
    run = te_host.Run(cfg)
    run.init_state()
    n = run.sJ * run.sK * run.nz
    col = np.linspace(0.5, 1.5, n).astype(np.float32) * np.float32(theta)
    for f in ("th", "th_a"):
        o = run.field_offset(f)
        run.upload(o, col.view(np.uint32))
        ref.M[o: o + n] = col.view(np.uint32)
    last = ref.names.index("ac_column")
    run.run(1, 0, last)
    run.sync()
    ref.prog.run(ref.M, 0, last)
    assert np.isfinite(ref.field("w")).all() and np.abs(ref.field("w")).max() > 0
    compare(run, ref)
    run.close()
