"""Far fields of many directions: the plan of the positions on an operator that
runs the row lists, positions beyond one group of records, dipoles that share a
position, device memory that leaves no room for the records, and what the first
call on a new operator costs. Each against a few directions at a time."""
import time

import numpy as np
import pytest

import dda_amd as D

from test_spare_buffers_gpu import Filled

pytestmark = pytest.mark.gpu


def _random_pol(ctx, op, k, seed):
    rng = np.random.default_rng(seed)
    p = rng.normal(size=(k, 3, op.vec_stride)) + 1j * rng.normal(size=(k, 3, op.vec_stride))
    p[:, :, op.nv:] = 0
    v = D.DeviceVector(ctx, k * op.vec_size, 64)
    v.upload(p.reshape(-1))
    return v


def _dirs(nq, seed=3):
    d = np.random.default_rng(seed).normal(size=(nq, 3))
    return d / np.linalg.norm(d, axis=1)[:, None]


def _few(op, pol, k, dirs, rhs):
    n = min(40, 7_000_000 // op.nv)  # the direct sums'
    return np.concatenate([D.far_field(op, pol, k, dirs[i:i + n], rhs[i:i + n]) for i in range(0, len(dirs), n)])


def _box(box, keep=None):
    z, y, x = np.meshgrid(*(np.arange(b) for b in box[::-1]), indexing="ij")
    k = keep(x, y, z) if keep else np.ones(x.shape, bool)
    return np.stack([a[k] for a in (x, y, z)], 1)


def _operator(ctx, pos, box, precision=32):
    return D.GpuMatVec(ctx, pos, None, box, 0.5e-6, 0.4 / 0.5e-6, nmat=1, precision=precision)


# phases of up to 200 radians and sums of up to 3 million terms: 1e-12 of the largest field
TOL = 1e-12


@pytest.mark.parametrize("box", [(30, 20, 20), (31, 21, 19), (1, 110, 90), (140, 9, 8), (2, 90, 60)])
def test_plan_from_row_lists(ctx, monkeypatch, box):
    print("box", box, flush=True)
    pos = _box(box, lambda x, y, z: (x + 2 * y + 3 * z) % 5 != 1)
    pos = pos[np.random.default_rng(5).permutation(len(pos))]
    cells = _operator(ctx, pos, box)
    monkeypatch.setenv("DDA_GENERIC_FFT", "1")
    rows = _operator(ctx, pos, box)
    pol = _random_pol(ctx, cells, 2, 1)
    nq = 8_000_000 // len(pos) + 100
    dirs, rhs = _dirs(nq), np.arange(nq) % 2
    a, b = (D.far_field(op, pol, 2, dirs, rhs) for op in (cells, rows))
    assert np.array_equal(a, b)  # the same segments, in the same order
    ref = _few(cells, pol, 2, dirs, rhs)
    assert np.abs(a - ref).max() <= TOL * np.abs(ref).max()
    for o in (cells, rows, pol):
        o.close()


def test_shared_positions(ctx):
    pos = _box((30, 20, 20))
    twice = np.concatenate([pos, pos[7:9]])
    op = _operator(ctx, twice, (30, 20, 20))
    pol = _random_pol(ctx, op, 1, 2)
    dirs = _dirs(900)
    got = D.far_field(op, pol, 1, dirs)
    ref = _few(op, pol, 1, dirs, np.zeros(900, int))
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()
    op.close()
    pol.close()


def test_groups_of_positions_and_no_room_for_records(ctx):
    """2.9 million dipoles, 1.5 million folded positions: two groups of records.
    Then the same call with 100 MB of device memory left, which its records do
    not fit: accepted all the same."""
    own = D.Context(0)  # without spare buffers of other tests
    box = (160, 136, 134)
    pos = _box(box)
    op = _operator(own, pos, box)
    pol = _random_pol(own, op, 2, 4)
    dirs = _dirs(200)
    rhs = np.arange(200) // 100
    ref = _few(op, pol, 2, dirs, rhs)
    with Filled(100 << 20) as f:
        print("left", f.left >> 20, "MB", flush=True)
        short = D.far_field(op, pol, 2, dirs, rhs)
    assert np.abs(short - ref).max() <= TOL * np.abs(ref).max()
    got = D.far_field(op, pol, 2, dirs, rhs)
    assert np.abs(got - ref).max() <= TOL * np.abs(ref).max()
    own.close()


def test_first_call_on_a_new_operator(ctx):
    """A program that evaluates one set of directions per particle pays for the
    plan each time: it has to stay within five times a later call (formed on the
    host it was 24 times one here)."""
    box = (200, 200, 200)
    pos = _box(box)
    times = []
    for _ in range(3):
        op = _operator(ctx, pos, box)
        pol = _random_pol(ctx, op, 1, 4) if not times else pol
        t = []
        for _ in range(4):
            ctx.synchronize()
            t0 = time.perf_counter()
            D.far_field(op, pol, 1, _dirs(64))
            t.append(time.perf_counter() - t0)
        times.append((t[0], min(t[1:])))
        op.close()
    print("first and later calls, us", [(round(a * 1e6), round(b * 1e6)) for a, b in times], flush=True)
    assert min(a for a, _ in times) <= 5 * min(b for _, b in times)
    pol.close()
