"""Blocks of right-hand sides whose passes leave out the rows outside the
planes' occupied ranges (where A1 is larger than 16 MB), against the oracle and,
bit for bit, against each right-hand side's own product, which works on every
row. Tolerances are those of the other matvec tests."""
import numpy as np
import pytest

import dda_amd as D
from dda_amd import problem as P

import cases

pytestmark = pytest.mark.gpu

RANGE_BYTES = 16 << 20
BOX = (60, 40, 8)


def _uses_ranges(op, nrhs):
    return bool(D.lib().dda_op_row_ranges(op.handle, nrhs))


def _particle(full):
    """Planes whose rows start late, end early, leave rows out, and one without
    any (full: every cell)."""
    rng = np.random.default_rng(17)
    z, y, x = np.meshgrid(*(np.arange(b) for b in BOX[::-1]), indexing="ij")
    keep = (rng.random(x.shape) < 0.5) & (y % 5 != 3) & (z != 4) & (y >= z) & ((y < 7) | (z != 2))
    if full:
        keep[:] = True
    return P.DipoleGeometry(np.stack([a[keep] for a in (x, y, z)], 1), None, [1.5 + 0.1j], 0.5e-6)


def _op(ctx, g, params, cs, precision, k):
    op = D.GpuMatVec(ctx, g.pos, g.mat, g.box, g.grid_unit, params.wave_num, precision=precision, grid=params.grid,
                     nmat=1)
    op.set_couple_constants_batch(np.array([cs * (1 + 0.1 * r) for r in range(k)]))
    return op


def _apply(ctx, op, v, conj=False):
    k = len(v)
    x = D.DeviceVector(ctx, k * op.vec_size, op.precision)
    y = D.DeviceVector(ctx, k * op.vec_size, op.precision)
    x.upload(np.asarray(v).reshape(-1))
    op.apply_batch(x, y, k, conj=conj)
    ctx.synchronize()
    out = y.download().reshape(k, -1)
    x.close()
    y.close()
    return out


# general and tuned plans on each axis, the longest planned Y axis, and one that
# only the run-time planned Y passes take (those work on every row)
@pytest.mark.parametrize("grid,ranges", [((120, 80, 16), True), ((128, 96, 32), True), ((126, 512, 20), True),
                                         ((128, 90, 18), True), ((120, 540, 16), False)])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("split", [0, 1])
def test_block_of_rows_with_gaps(ctx, grid, ranges, precision, split):
    """After a product of NaNs of the whole box in the same buffers, then one of
    the particle's own. The block runs whole or as two halves on two streams, of
    which only the first and larger one is beyond the limit."""
    csz = precision // 4
    per = 3 * BOX[1] * BOX[2] * (-(-grid[0] // (128 // csz)) * 128)
    h = RANGE_BYTES // per + 1
    k = 2 * h - 1 if split else h
    print("grid", grid, "precision", precision, "split", split, "right-hand sides", k, flush=True)
    g = _particle(False)
    params = P.DDAParams(g, 6e-6, grid)
    cs = P.couple_constants(params, *P.beam_pols((0.3, -0.2, 0.8))[:2])[1]
    gf = _particle(True)
    pf = P.DDAParams(gf, 6e-6, grid)
    bad = _op(ctx, gf, pf, cs, precision, k)
    _apply(ctx, bad, np.full((k, pf.vec_size), np.nan + 0j))
    bad.close()
    op = _op(ctx, g, params, cs, precision, k)
    op.variants([-1] * 5 + [split])
    assert _uses_ranges(op, h) == ranges and not _uses_ranges(op, h - 1)
    _apply(ctx, op, np.full((k, params.vec_size), np.nan + 0j))
    v = np.array([P.random_dipole_vector(params, seed=4 + r) for r in range(k)])
    for conj in (False, True):
        got = _apply(ctx, op, v, conj)
        for r in sorted({0, h - 1, min(h, k - 1), k - 1}):
            ref = cases.oracle_problem(g, params, cs * (1 + 0.1 * r), dmat_precision=64)
            assert cases.rel_err(got[r], ref.matvec(v[r], conj=conj, precision=64)) <= (1e-12 if precision == 64 else 1e-5)
        for r in range(k):  # alone: with right-hand side r's constants in first place
            op.set_couple_constants(cs * (1 + 0.1 * r))
            assert np.array_equal(_apply(ctx, op, v[r:r + 1], conj)[0], got[r]), r
        op.set_couple_constants_batch(np.array([cs * (1 + 0.1 * r) for r in range(k)]))
    op.close()


@pytest.mark.parametrize("grid,nrhs,y_tiles,z_tile", [((128, 96, 64), 32, True, True), ((128, 96, 48), 64, True, True),
                                                      ((64, 96, 64), 64, True, False), ((128, 96, 32), 32, False, True)])
def test_large_blocks_take_other_tiles(ctx, grid, nrhs, y_tiles, z_tile):
    """FP32 blocks that the untuned rule gives 64-column tiles in the Y and Z
    passes: against the oracle, and bit for bit each right-hand side's own
    product with the tiles of a single one. (y_tiles, z_tile: what the rule says
    of the block; a single right-hand side gets neither.)"""
    gx, gy, gz = grid
    box = (gx // 2, gy // 2 - 3, gz // 2)
    print("grid", grid, "right-hand sides", nrhs, flush=True)
    # (as default_col_variant and wide_z_tile have it)
    assert (gx % 64 == 0 and (gx // 64) * 3 * box[2] * nrhs >= 6144) == y_tiles
    assert (gx % 128 == 0 and (gx // 64) * gy * nrhs >= 6144) == z_tile
    g = P.ellipsoid(*(b / 2 for b in box), 1.33 + 0.01j, 0.5e-6)
    params = P.DDAParams(g, 6e-6, grid)
    cs = P.couple_constants(params, *P.beam_pols((0.3, -0.2, 0.8))[:2])[1]
    op = _op(ctx, g, params, cs, 32, nrhs)
    v = np.array([P.random_dipole_vector(params, seed=4 + r) for r in range(nrhs)])
    got = _apply(ctx, op, v)
    for r in (0, nrhs // 2, nrhs - 1):
        ref = cases.oracle_problem(g, params, cs * (1 + 0.1 * r), dmat_precision=64)
        assert cases.rel_err(got[r], ref.matvec(v[r], precision=64)) <= 1e-5
    for r in range(0, nrhs, 5):
        op.set_couple_constants(cs * (1 + 0.1 * r))
        assert np.array_equal(_apply(ctx, op, v[r:r + 1])[0], got[r]), r
    op.close()
