"""The tuner keeps a pass on the untuned rule (-1) unless another variant beats
the one that the rule picks by more than 2%: checked against the timings in its
own report, on grids where the rule picks each of its variants."""
import ctypes
import re

import numpy as np
import pytest

import dda_amd as D

pytestmark = pytest.mark.gpu

PASSES = ["Y forward", "Z + tensor", "Y inverse", "X forward", "X inverse"]


# (grid, precision, what the rule picks for Y and for Z with one right-hand side)
@pytest.mark.parametrize("grid,precision,y,z", [((1024, 128, 256), 32, 5, 1), ((1024, 512, 64), 32, 0, 3),
                                                ((256, 64, 64), 32, 1, 1), ((64, 64, 512), 32, 1, 2),
                                                ((64, 96, 64), 64, 0, 0)])
def test_tuner_keeps_the_untuned_rule(ctx, grid, precision, y, z):
    print("grid", grid, "precision", precision, flush=True)
    box = [n // 2 for n in grid]
    rng = np.random.default_rng(2)
    pos = np.unique(np.stack([rng.integers(0, b, 3000) for b in box], 1), axis=0)
    op = D.GpuMatVec(ctx, pos, None, box, 0.5e-6, 1e6, precision=precision, grid=grid, nmat=1)
    op.set_couple_constants(np.ones((1, 3)) * 1e-10)
    buf = ctypes.create_string_buffer(8192)
    assert D.lib().dda_op_tune(op.handle, 1, buf, 8192) == D.OK
    report = buf.value.decode()
    print(report, flush=True)
    got = op.variants()[:5]
    for i, (name, rule) in enumerate(zip(PASSES, (y, z, y, 0, 0))):
        line = re.search(re.escape(name) + r": (.*?) ->", report).group(1)
        t = [float(v) for v in re.findall(r" ([\d.]+) us", line)]
        best = int(np.argmin(t))
        # (the report's figures are rounded to 0.1 us)
        if t[best] - 0.05 > 0.98 * (t[rule] + 0.05):
            assert got[i] == -1, (name, got[i])
        elif t[best] + 0.05 < 0.98 * (t[rule] - 0.05):
            assert got[i] >= 0 and t[got[i]] <= t[best] + 0.1, (name, got[i])
    op.close()
