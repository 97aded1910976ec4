"""kernel_variant 2: the sweeps with the z-face statements of the stress phase
left to their own launch (and so no fused step), the bits of variants 0 and 1."""
import numpy as np
import pytest

from opesci.backend import Context
from workloads import box_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,order,het,double,storage", [
    ((17, 14, 66), 4, False, False, 'native'), ((13, 12, 20), 4, True, False, 'native'),
    ((12, 15, 70), 2, False, True, 'native'), ((15, 16, 33), 8, True, False, 'bf16')])
def test_variant_2_leaves_the_z_faces_out(sizes, order, het, double, storage):
    g, _ = box_model(sizes, order, 7, hetero=het, double=double, storage=storage)
    plan = g.lower()
    out = []
    for variant in (0, 1, 2):
        plan.kernel_variant = variant
        plan.fuse_step = variant == 2
        with Context(plan) as ctx:
            deep, launches, applied = ctx.stats(full=True)[1:4]
            assert deep > 0 and applied == int(variant == 0) and launches == int(variant != 0)
            assert ctx.fused_margin() == 0
            ctx.init()
            ctx.run()
            out.append(ctx.fields())
    for f in range(9):
        assert np.array_equal(out[2][f], out[0][f]) and np.array_equal(out[2][f], out[1][f]), f
