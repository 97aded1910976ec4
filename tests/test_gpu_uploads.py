"""Steps after an upload: a step keeps its launches unless the upload touched
cells whose zeros steps leave out (a velocity, where some statement is left
out), and its bits are those of every statement as a launch of its own
(kernel_variant 1) either way, alone and in a batch."""
import numpy as np
import pytest

from opesci.backend import Context
from opesci.batch import Batch
from workloads import box_model

pytestmark = pytest.mark.gpu


def noise(ctx, plan, fields, seed):
    rng = np.random.default_rng(seed)
    dtype = np.float64 if plan.real_bytes == 8 else np.float32
    for f in fields:
        for lvl in (0, 1):
            ctx.upload(f, lvl, rng.standard_normal(plan.dims).astype(dtype))


def levels(ctx):
    return [ctx.download(f, lvl) for f in range(9) for lvl in (0, 1)]


@pytest.mark.parametrize("order,double,fields,full", [
    (4, False, (0, 2, 5), 0), (2, True, (3, 8), 0), (8, False, (4, 6, 7), 0), (6, False, (1,), 2), (2, False, (0, 3), 2)])
def test_steps_after_an_upload(order, double, fields, full):
    plan = box_model((12, 11, 13), order, 9, double=double)[0].lower()
    out = []
    for variant in (0, 1):
        plan.kernel_variant = variant
        with Context(plan) as ctx:
            ctx.init()
            ctx.run(3)
            short = ctx.stats()[0]
            noise(ctx, plan, fields, 5)
            if variant == 0:
                for left in range(full, 0, -1):
                    assert ctx.stats()[0] > short, left
                    ctx.run(1)
                assert ctx.stats()[0] == short
            ctx.run(6 - (full if variant == 0 else 0))
            out.append(levels(ctx))
    for i, (u, v) in enumerate(zip(*out)):
        assert np.array_equal(u, v), (i // 2, i % 2)


def test_batch_after_uploads_at_odd_steps():
    plans = [box_model(s, o, 9)[0].lower() for s, o in (((9, 11, 8), 2), ((10, 9, 12), 4), ((11, 10, 10), 8))]
    out = []
    for variant in (0, 1):
        for p in plans:
            p.kernel_variant = variant
        with Batch(plans, tune=False) as b:
            assert b.run(1) > 0
            for i, (c, p) in enumerate(zip(b.contexts, plans)):
                noise(c, p, (i, 3 + i), i)
            assert b.run(1) > 0
            assert b.run(5) > 0
            assert [c.steps() for c in b.contexts] == [7, 7, 7]
            out.append([x for c in b.contexts for x in levels(c)])
    for u, v in zip(*out):
        assert np.array_equal(u, v)
