"""Boundary statements as pieces (cut into rectangles, velocities along an
axis evaluated inside the statements across it) against every statement in
its hazard level (kernel_variant 1), bit for bit on both time levels."""
import numpy as np
import pytest

from opesci.backend import Context
from workloads import box_model

pytestmark = pytest.mark.gpu


def run(plan, variant):
    plan.kernel_variant = variant
    with Context(plan) as ctx:
        launches = ctx.stats()[0]
        ctx.init()
        ctx.run(9)
        return launches, [ctx.download(f, lvl) for f in range(9) for lvl in (0, 1)]


@pytest.mark.parametrize("sizes,order,het,double,storage", [
    # 4th order: cuts that meet or cross, edges longer than a block, both
    # media, coefficients per point and rounding to storage in place
    ((6, 6, 6), 4, False, False, 'native'), ((7, 5, 6), 4, True, False, 'native'),
    ((8, 7, 9), 4, True, True, 'native'), ((9, 10, 11), 4, False, False, 'fp16'),
    ((11, 9, 10), 4, True, False, 'bf16'), ((17, 40, 33), 4, True, False, 'native'),
    ((40, 18, 70), 4, True, False, 'fp16'), ((70, 33, 20), 4, False, True, 'native'),
    ((5, 4, 5), 2, True, False, 'native'), ((30, 21, 70), 2, False, False, 'bf16'),
    ((9, 8, 8), 6, True, False, 'native'), ((33, 20, 17), 6, False, False, 'native'),
    ((11, 10, 12), 8, True, False, 'native'), ((26, 31, 40), 8, False, True, 'native')])
def test_pieces_equal_levels(sizes, order, het, double, storage):
    g, _ = box_model(sizes, order, 12, hetero=het, double=double, storage=storage)
    plan = g.lower()
    n, a = run(plan, 0)
    levels, b = run(plan, 1)
    assert n < levels
    if order == 4:
        assert n == 5
    for i, (u, v) in enumerate(zip(a, b)):
        assert np.array_equal(u, v, equal_nan=True), (i // 2, i % 2)
