"""The deep z-face statements of the stress phase in the stress sweep, for the
types, media and z sizes it takes them for by default, against the same plan
with every statement as a launch of its own (kernel_variant 1), bit for bit
on both time levels."""
import numpy as np
import pytest

from opesci.backend import Context
from workloads import box_model

pytestmark = pytest.mark.gpu


def run(plan, variant, tile_y=0):
    plan.kernel_variant, plan.tile_y = variant, tile_y
    with Context(plan) as ctx:
        applied = ctx.stats(full=True)[3]
        ctx.init()
        ctx.run(7)
        return applied, [ctx.download(f, lvl) for f in range(9) for lvl in (0, 1)]


@pytest.mark.parametrize("sizes,order,het,double,storage,tile_y", [
    # read path, 4th order: both faces in one tile (few and most columns, more
    # coefficients than points), a face in each of several, 16-bit storage
    ((13, 12, 9), 4, True, False, 'native', 0), ((12, 35, 16), 4, True, False, 'native', 0),
    ((12, 19, 72), 4, True, False, 'native', 0), ((11, 23, 73), 4, True, True, 'native', 4),
    ((14, 17, 130), 4, True, False, 'fp16', 0), ((12, 18, 65), 4, True, False, 'bf16', 8),
    # other orders and FP64, high faces right behind a multiple of 128
    ((9, 11, 64), 2, True, True, 'native', 0), ((14, 13, 66), 6, True, False, 'fp16', 0),
    ((15, 16, 129), 8, True, False, 'native', 0), ((11, 12, 129), 2, False, True, 'native', 0),
    ((12, 14, 128), 4, False, True, 'native', 0), ((13, 12, 129), 4, False, False, 'native', 0),
    ((12, 13, 130), 4, False, False, 'fp16', 0)])
def test_z_faces_in_sweep(sizes, order, het, double, storage, tile_y):
    g, _ = box_model(sizes, order, 9, hetero=het, double=double, storage=storage)
    plan = g.lower()
    applied, a = run(plan, 0, tile_y)
    none, b = run(plan, 1)
    assert (applied, none) == (1, 0)
    for i, (u, v) in enumerate(zip(a, b)):
        assert np.array_equal(u, v, equal_nan=True), (i // 2, i % 2)
