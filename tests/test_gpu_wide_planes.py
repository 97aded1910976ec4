"""Boundary launches with more points than blocks that fit the chip hold (2048
blocks of 256): a thread then takes several points of a statement of at most one
term, up to eight in two rounds, with a ragged tail.  Against every statement in
its hazard level (kernel_variant 1), bit for bit on both time levels."""
import numpy as np
import pytest

from opesci.backend import Context
from workloads import box_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,storage,double", [
    # 24 statements on the z faces: 2.2 million points, eight per thread; 1.0 million, four
    ((300, 301, 9), 'fp16', False), ((211, 198, 9), 'native', True)])
def test_many_points_per_thread(sizes, storage, double):
    g, _ = box_model(sizes, 8, 3, storage=storage, double=double)
    g.fuse_boundary = False   # the z faces stay boundary launches
    plan = g.lower()
    out = []
    for variant in (0, 1):
        plan.kernel_variant = variant
        with Context(plan) as ctx:
            ctx.init()
            ctx.run()
            out.append([ctx.download(f, lvl) for f in range(9) for lvl in (0, 1)])
    assert all(np.abs(x).max() > 0 for x in out[0])
    for i, (u, v) in enumerate(zip(*out)):
        assert np.array_equal(u, v, equal_nan=True), (i // 2, i % 2)
