"""The matvec on grid lengths that run a general plan (two or three stages of
unequal radices, some threads without a butterfly), each length on the X, the
Y and the Z axis, against the oracle.

The box spans half the long axis, less one cell for every second length (an
odd number of padded points), and a few cells of the 16-point axes, so that a
length's first and last kept points, partial column tiles and partly filled
work-groups all occur. Tolerances are those of the other matvec tests: 1e-12
in FP64 and 1e-5 in FP32."""
import numpy as np
import pytest

import dda_amd as D
from dda_amd import problem as P

import cases

pytestmark = pytest.mark.gpu

LENGTHS = [8, 10, 12, 14, 16, 18, 20, 24, 28, 30, 36, 40, 42, 50, 54, 56, 60, 70, 72, 80, 84, 90, 98, 100, 108, 112,
           120, 126, 140, 144, 150, 160, 162, 168, 180, 196, 200, 210, 216, 224, 240, 250, 252, 270, 280, 288, 294,
           300, 320, 324, 336, 350, 360, 378, 384, 392, 400, 420, 432, 448, 450, 480, 486, 490, 500, 504]


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("n", LENGTHS)
def test_matvec_general_lengths(ctx, n, axis):
    print("length", n, "axis", axis, flush=True)
    box, grid = [5, 4, 3], [16, 16, 16]
    box[axis] = n // 2 - (LENGTHS.index(n) % 2)
    grid[axis] = n
    g = P.box(*box, 1.5 + 0.1j, 0.5e-6)
    g.mat = (np.arange(g.nv) % 3 == 0).astype(np.uint8)
    g.materials = [1.5 + 0.1j, 1.3 + 0.2j]
    params = P.DDAParams(g, 6e-6, grid)
    assert params.grid == tuple(grid)
    prop, pol, _ = P.beam_pols((0.3, -0.2, 0.8))
    cc, cs = P.couple_constants(params, prop, pol)
    orc = cases.oracle_problem(g, params, cs, dmat_precision=64)
    x = P.random_dipole_vector(params, seed=n)
    for conj in (False, True):
        y_ref = orc.matvec(x, conj=conj, precision=64)
        for precision, tol in ((64, 1e-12), (32, 1e-5)):
            op = D.GpuMatVec(ctx, g.pos, g.mat, g.box, g.grid_unit, params.wave_num, precision=precision,
                             grid=params.grid, nmat=2)
            op.set_couple_constants(cs)
            y = D.MatVecGpu(op).apply(x, conj=conj)
            assert cases.rel_err(y, y_ref) <= tol
            assert np.all(y[params.nv:params.vec_stride] == 0)
            op.close()
