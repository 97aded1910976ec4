"""Models whose off-axis coefficients of the normal stresses differ (the C ABI
takes any): the stress sweep with a sum per stress and axis, and the z faces in
it, against the gather kernels (kernel_variant 1), bit for bit."""
import numpy as np
import pytest

from opesci.backend import Context
from workloads import box_model

pytestmark = pytest.mark.gpu


def general(sizes, order, **kw):
    plan = box_model(sizes, order, 7, **kw)[0].lower()
    cn = np.array(plan.cn)
    cn[0, 1] *= 1.25
    cn[2, 0] *= 0.875
    cn[1, 2, 0] *= 1.125
    plan.cn = cn
    return plan


@pytest.mark.parametrize("sizes,order,kw", [
    ((13, 17, 66), 4, {}), ((12, 14, 20), 4, dict(hetero=True, storage='bf16')), ((11, 12, 73), 2, dict(double=True)),
    ((14, 13, 64), 6, dict(storage='fp16')), ((15, 16, 30), 8, dict(hetero=True)), ((12, 13, 19), 4, dict(double=True)),
    ((9, 10, 33), 2, {})])
def test_general_coefficients(sizes, order, kw):
    plan = general(sizes, order, **kw)
    out = []
    for variant in (0, 1):
        plan.kernel_variant = variant
        with Context(plan) as ctx:
            assert ctx.stats(full=True)[3] == 1 - variant
            ctx.init()
            ctx.run()
            out.append([ctx.download(f, lvl) for f in range(9) for lvl in (0, 1)])
    assert np.isfinite(out[0]).all() and np.abs(out[0]).max() > 0
    for i, (u, v) in enumerate(zip(*out)):
        assert np.array_equal(u, v), (i // 2, i % 2)


def test_general_coefficients_in_the_fused_step():
    plan = general((40, 33, 70), 4)
    out = []
    for fuse in (True, False):
        plan.fuse_step = fuse
        with Context(plan) as ctx:
            assert (ctx.fused_margin() > 0) == fuse
            ctx.init()
            ctx.run()
            out.append(ctx.fields())
    for f in range(9):
        assert np.array_equal(out[0][f], out[1][f]), f
