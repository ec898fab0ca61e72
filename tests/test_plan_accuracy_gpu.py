"""How far FP64 products on general plans are from the exact ones (the oracle in
long double), against the run-time planned kernels' (radices up to 8) on the same
vectors. The root mean square over four vectors of a product, of 10^4 and more
rounding errors each, repeats to a percent or two: 5% are allowed."""
import numpy as np
import pytest

import dda_amd as D
from dda_amd import problem as P

import cases

pytestmark = pytest.mark.gpu

# grids of cubes of half the length, and of long boxes on each axis
GRIDS = [(18, 18, 18), (56, 56, 56), (80, 80, 80), (112, 28, 28), (20, 384, 20), (20, 28, 224), (336, 20, 20)]


@pytest.mark.parametrize("grid", GRIDS)
def test_error_no_larger_than_run_time_planned(ctx, monkeypatch, grid):
    g = P.box(*(n // 2 for n in grid), 1.5 + 0.1j, 0.5e-6)
    params = P.DDAParams(g, 6e-6, grid)
    assert params.grid == grid
    cs = P.couple_constants(params, *P.beam_pols((0.3, -0.2, 0.8))[:2])[1]
    orc = cases.oracle_problem(g, params, cs)
    v = [P.random_dipole_vector(params, seed=s) for s in range(4)]
    ref = [orc.matvec(x, precision=80) for x in v]
    err = {}
    for generic in (False, True):
        if generic:
            monkeypatch.setenv("DDA_GENERIC_FFT", "1")
        op = D.GpuMatVec(ctx, g.pos, None, g.box, g.grid_unit, params.wave_num, grid=grid, nmat=1)
        op.set_couple_constants(cs)
        mv = D.MatVecGpu(op)
        err[generic] = np.sqrt(np.mean([cases.rel_err(np.asarray(mv.apply(x)), y) ** 2 for x, y in zip(v, ref)]))
        op.close()
    print("grid", grid, "general %.3e run-time planned %.3e" % (err[False], err[True]), flush=True)
    assert err[False] <= 1.05 * err[True]
