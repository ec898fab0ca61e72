"""The buffers of destroyed operators that a context keeps for its next ones:
given back wherever the library finds the device's memory short, reused without
one operator's work reaching another's, also from several threads and after
products on a stream of the caller's."""
import ctypes
import threading

import numpy as np
import pytest

import dda_amd as D
from dda_amd import problem as P

pytestmark = pytest.mark.gpu

BOX = (96, 96, 96)


def _operator(ctx, box, precision=64, nrhs=1, **kw):
    z, y, x = np.meshgrid(*(np.arange(b) for b in box[::-1]), indexing="ij")
    g = P.DipoleGeometry(np.stack([a.ravel() for a in (x, y, z)], 1), None, [1.5 + 0.1j], 0.5e-6)
    params = P.DDAParams(g, 6e-6)
    cs = P.couple_constants(params, *P.beam_pols((0.3, -0.2, 0.8))[:2])[1]
    op = D.GpuMatVec(ctx, g.pos, None, g.box, g.grid_unit, params.wave_num, precision=precision, grid=params.grid,
                     nmat=1, **kw)
    op.set_couple_constants_batch(np.array([cs] * nrhs))
    return op, params


class Filled:
    """The device's memory taken up to `leave` bytes (not through the library,
    which would give the spare buffers back)."""

    def __init__(self, leave):
        self.blocks = []
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        for _ in range(64):
            assert D.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            if free.value <= leave + (8 << 20):
                break
            p = ctypes.c_void_p()
            assert D.lib().hipMalloc(ctypes.byref(p), ctypes.c_size_t(free.value - leave)) == 0
            self.blocks.append(p)
        self.left = free.value

    def __enter__(self):
        return self

    def __exit__(self, *exc):
        for p in self.blocks:
            D.lib().hipFree(p)


@pytest.mark.parametrize("what", ["malloc of another context", "solver"])
def test_spare_buffers_are_given_back(what):
    own, other = D.Context(0), D.Context(0)
    keep, _ = _operator(own, BOX)
    gone, _ = _operator(own, BOX, nrhs=2)  # leaves 850 MB
    gone.close()
    with Filled(100 << 20) as f:
        print(what, "left", f.left >> 20, "MB", flush=True)
        if what == "solver":  # 340 MB of vectors
            D.GpuQmrCs(keep).close()
        else:
            D.DeviceVector(other, 25_000_000, 64).close()
    keep.close()
    own.close()
    other.close()


def _product(ctx, op, params, seed):
    x = D.DeviceVector(ctx, op.vec_size, op.precision)
    y = D.DeviceVector(ctx, op.vec_size, op.precision)
    x.upload(P.random_dipole_vector(params, seed=seed))
    op.apply(x, y)
    ctx.synchronize()
    out = y.download()
    x.close()
    y.close()
    return out


SHAPES = [((24, 20, 16), 64), ((23, 21, 16), 64), ((30, 22, 18), 32), ((25, 20, 17), 32)]


def _expected():
    out = []
    for q, (box, precision) in enumerate(SHAPES):
        fresh = D.Context(0)
        op, params = _operator(fresh, box, precision)
        out.append(_product(fresh, op, params, q))
        op.close()
        fresh.close()
    return out


def test_operators_in_each_others_buffers():
    want = _expected()
    own = D.Context(0)
    for rep in range(3):
        for q in np.random.default_rng(rep).permutation(len(SHAPES)):
            op, params = _operator(own, *SHAPES[q])
            assert np.array_equal(_product(own, op, params, int(q)), want[q]), (rep, q)
            op.close()
    own.close()


def test_threads_that_share_a_context():
    """Distinct operators of one context, each used by one thread."""
    want = _expected()
    own = D.Context(0)
    bad = []

    def work(q):
        try:
            for _ in range(6):
                op, params = _operator(own, *SHAPES[q])
                if not np.array_equal(_product(own, op, params, q), want[q]):
                    bad.append(q)
                op.close()
        except Exception as e:  # noqa: BLE001 (shown by the assertion)
            bad.append(e)

    threads = [threading.Thread(target=work, args=(q,)) for q in range(len(SHAPES))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    own.close()
    assert not bad


def test_products_on_a_callers_stream():
    """An operator destroyed while its products wait on the caller's stream: the
    next operator of the shape works on the context's stream beside them."""
    own = D.Context(0)
    box = (96, 90, 80)
    op, params = _operator(own, box)
    x = [D.DeviceVector(own, op.vec_size, 64) for _ in range(2)]
    y = [D.DeviceVector(own, op.vec_size, 64) for _ in range(2)]
    for q in range(2):
        x[q].upload(P.random_dipole_vector(params, seed=q))
    op.apply(x[0], y[0])
    op.apply(x[1], y[1])
    own.synchronize()
    want = [v.download() for v in y]
    st = ctypes.c_void_p()
    assert D.lib().hipStreamCreateWithFlags(ctypes.byref(st), 1) == 0  # non-blocking
    for _ in range(40):
        op.apply(x[0], y[0], stream=st)
    op.close()
    nxt, _ = _operator(own, box)
    for _ in range(10):
        nxt.apply(x[1], y[1])
    own.synchronize()
    assert D.lib().hipStreamSynchronize(st) == 0
    assert np.array_equal(y[0].download(), want[0]) and np.array_equal(y[1].download(), want[1])
    nxt.close()
    assert D.lib().hipStreamDestroy(st) == 0
    for v in x + y:
        v.close()
    own.close()


def _device_bytes(op):
    n = ctypes.c_size_t()
    assert D.lib().dda_op_info(op.handle, None, None, ctypes.byref(n)) == D.OK
    return n.value


def _free():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert D.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def test_a_larger_buffer_counts_as_it_is():
    fresh, own = D.Context(0), D.Context(0)
    op, _ = _operator(fresh, (96, 96, 80))
    alone = _device_bytes(op)
    op.close()
    _operator(own, BOX)[0].close()  # its buffers are a fifth larger
    op, _ = _operator(own, (96, 96, 80))
    assert 1.15 * alone <= _device_bytes(op) <= 1.25 * alone
    op.close()
    own.close()
    fresh.close()


def test_spare_buffers_stay_within_a_gigabyte():
    """One operator of more than that, then eight of 340 MB that are destroyed
    together; all of it is given back with the context."""
    own = D.Context(0)
    before = _free()
    small, _ = _operator(own, (40, 40, 40))
    small.close()
    kept = _free()
    big, _ = _operator(own, (128, 128, 128), nrhs=2)  # grid buffers of 1.2 GB and 600 MB
    big.close()
    assert before - _free() <= (1 << 30) + (64 << 20)
    ops = [_operator(own, BOX)[0] for _ in range(8)]
    assert before - _free() >= 8 * (300 << 20)
    for op in ops:
        op.close()
    assert before - _free() <= (1 << 30) + (64 << 20)
    own.close()
    assert _free() >= kept - (64 << 20)


def test_buffers_that_fit_outlast_those_too_large():
    """A large block's buffers first serve smaller operators, whose own set then
    fits the limit: once it is made, destroying and making such an operator again
    frees nothing (a hipFree of the buffers takes most of a millisecond)."""
    own = D.Context(0)
    op, _ = _operator(own, (64, 48, 32), 32, nrhs=128)  # grid buffers of 300 and 600 MB
    op.close()
    for _ in range(3):
        op, _ = _operator(own, (128, 128, 128), 32, nrhs=2)  # 100, 200, 200, 400 and 100 MB
        op.close()
    kept = _free()
    for _ in range(3):
        op, _ = _operator(own, (128, 128, 128), 32, nrhs=2)
        # positions, materials and cell map, 17 bytes a cell of the full box, in pages of
        # 2 MB, and small arrays: no grid buffer (100 MB and more) was taken anew
        assert kept - _free() <= 17 * op.nv + (16 << 20)
        op.close()
        assert abs(kept - _free()) <= 16 << 20
    own.close()
