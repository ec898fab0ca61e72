"""The interaction tensor formed by octants (planned lengths on every axis)
against the whole-grid transforms of the run-time planned kernels
(DDA_GENERIC_FFT=1), component by component.

Both are double precision transforms of the same values, some tens of
roundings deep: 1e-13 of a component's largest entry. In single precision
(stored rounded) they may round to neighbours: 2^-23 of it."""
import numpy as np
import pytest

import dda_amd as D
from dda_amd import problem as P

pytestmark = pytest.mark.gpu

# box, grid: shortest and longest planned lengths on each axis, lengths of two
# and three stages, boxes of half the grid (offset G/2 - 1 in use), less and one cell
CASES = [((4, 5, 3), (8, 10, 8)), ((1, 2, 1), (8, 8, 12)), ((512, 3, 2), (1024, 8, 8)), ((2, 512, 3), (8, 1024, 10)),
         ((3, 2, 512), (10, 8, 1024)), ((250, 4, 7), (500, 16, 14)), ((5, 245, 4), (14, 490, 8)),
         ((3, 4, 161), (8, 12, 392)), ((23, 18, 30), (48, 36, 64)), ((40, 35, 27), (80, 70, 54))]


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("box,grid", CASES)
def test_octant_tensor_matches_whole_grid(ctx, monkeypatch, box, grid, precision):
    print("box", box, "grid", grid, "precision", precision, flush=True)
    pos = np.array([[0, 0, 0], [b - 1 for b in box]]) if max(box) > 1 else np.zeros((1, 3), int)

    def tensor():
        op = D.GpuMatVec(ctx, pos, None, box, 0.5e-6, 1e6, precision=precision, grid=grid, nmat=1)
        dm = op.dmatrix()
        op.close()
        return dm

    got = tensor()
    monkeypatch.setenv("DDA_GENERIC_FFT", "1")
    ref = tensor()
    tol = 1e-13 if precision == 64 else 2.0 ** -23
    for c in range(6):
        scale = np.abs(ref[..., c]).max()
        assert np.abs(got[..., c] - ref[..., c]).max() <= tol * scale
