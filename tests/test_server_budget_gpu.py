"""What the job server counts for a job against the operators that its solve
makes: every buffer of both precisions is in the footprint."""
import ctypes

import numpy as np
import pytest

import dda_amd as D
from dda_amd import serving as S

pytestmark = pytest.mark.gpu


def _device_bytes(op):
    n = ctypes.c_size_t()
    assert D.lib().dda_op_info(op.handle, None, None, ctypes.byref(n)) == D.OK
    return n.value


# a sphere, a flat and a long box: rows of odd lengths, many rows, few dipoles to a cell map
@pytest.mark.parametrize("shape,dim,other", [("sphere", 33, None), ("box", 13, (61, 5)), ("ellipsoid", 70, (9, 20))])
@pytest.mark.parametrize("solver,mixed", [("bicgstab", True), ("qmr", True), ("qmr", False)])
def test_footprint_covers_the_operators(shape, dim, other, solver, mixed):
    rng = np.random.default_rng(3)
    job = S.make_job(rng, shape, dim, 1.4 + 0.02j, **({"other": other} if other else {}))
    srv = D.Server(slots=1, solver=solver, mixed=mixed, eps=1e-4)
    res = srv.wait(S.submit(srv, job))[2]
    srv.close()
    ctx = D.Context(0)
    cache = D.TensorCache(ctx, 1 << 30)
    g, params = job.geometry, job.params
    grid = [D.lib().dda_fft_fit_static(2 * int(b)) for b in g.box]  # the server's choice
    k = len(job.cc_sqrt)
    need = 0
    for precision in (64, 32) if mixed else (64,):
        op = D.GpuMatVec(ctx, g.pos, g.mat, g.box, g.grid_unit, params.wave_num, precision=precision,
                         grid=grid, nmat=len(g.materials), cache=cache)
        op.set_couple_constants_batch(job.cc_sqrt)
        need += _device_bytes(op)
        op.close()
    # the Krylov vectors: eight in the iteration's precision, and in FP64 six of the
    # refinement and eight more of a Lanczos method's fallback
    n = 3 * params.vec_stride * k
    need += n * (8 * 8 + 6 * 16 + (8 * 16 if solver == "qmr" else 0)) if mixed else n * 12 * 16
    ctx.close()
    print(shape, "grid", grid, "footprint", res["footprint"], "needed", need, flush=True)
    assert need <= res["footprint"] <= 1.25 * need
