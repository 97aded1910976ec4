"""A step without the velocity statements that store zeros over zeros (and with
the last-plane zeros in the velocity sweep) against the same step with every
statement as a launch of its own (kernel_variant 1), bit for bit on both time
levels: after an init, and after uploads that leave anything in the ghosts."""
import numpy as np
import pytest

from opesci.backend import Context
from opesci.batch import Batch
from workloads import box_model

pytestmark = pytest.mark.gpu

FIELDS = 9


def levels(ctx):
    return [ctx.download(f, lvl) for f in range(FIELDS) for lvl in (0, 1)]


def upload_noise(ctx, plan, seed):
    rng = np.random.default_rng(seed)
    dtype = np.float64 if plan.real_bytes == 8 else np.float32
    for f in range(FIELDS):
        for lvl in (0, 1):
            ctx.upload(f, lvl, rng.standard_normal(plan.dims).astype(dtype))


def run(plan, variant, pieces, noise):
    """init, pieces[0] steps, an upload when `noise`, the other pieces"""
    plan.kernel_variant = variant
    with Context(plan) as ctx:
        ctx.init()
        ctx.run(pieces[0])
        if noise:
            upload_noise(ctx, plan, 3)
        for n in pieces[1:]:
            ctx.run(n)
        return levels(ctx)


@pytest.mark.parametrize("sizes,order,het,double,storage", [
    ((9, 11, 8), 2, False, False, 'native'), ((8, 9, 70), 2, True, True, 'native'),
    ((12, 9, 10), 4, False, False, 'native'), ((13, 8, 66), 6, False, True, 'native'),
    ((9, 10, 11), 6, False, False, 'fp16'), ((9, 17, 69), 8, True, False, 'bf16'), ((10, 9, 64), 8, True, False, 'native')])
@pytest.mark.parametrize("pieces,noise", [((5,), False), ((2, 1, 4), True), ((3, 6), True)])
def test_step_equals_every_statement(sizes, order, het, double, storage, pieces, noise):
    g, _ = box_model(sizes, order, 9, hetero=het, double=double, storage=storage)
    plan = g.lower()
    a = run(plan, 0, pieces, noise)
    b = run(plan, 1, pieces, noise)
    for i, (u, v) in enumerate(zip(a, b)):
        assert np.array_equal(u, v, equal_nan=True), (i // 2, i % 2)


def test_step_keeps_statements_with_terms():
    """one ghost plane of U takes values instead of zeros: its statement and
    every zero statement that meets it stay"""
    g, _ = box_model((11, 12, 13), 6, 6)
    plan = g.lower()
    st = plan.stmts
    ghost = next(i for i, s in enumerate(st) if s['phase'] == 3 and s['field'] == 0 and s['axis'] == 0 and s['plane'] == 1)
    image = next(s for s in st if s['phase'] == 2 and s['field'] == 3 and s['axis'] == 0 and s['nterms'] == 1)
    st['nterms'][ghost], st['term0'][ghost] = 1, image['term0']
    a = run(plan, 0, (6,), False)
    b = run(plan, 1, (6,), False)
    assert np.abs(a[0][1]).max() > 0.0
    for u, v in zip(a, b):
        assert np.array_equal(u, v)


def test_batch_after_upload():
    plans = [box_model(s, o, 6, hetero=h)[0].lower() for s, o, h in
             (((9, 11, 8), 2, False), ((10, 9, 12), 6, True), ((8, 9, 10), 8, False))]
    out = []
    for variant in (0, 1):
        for p in plans:
            p.kernel_variant = variant
        with Batch(plans, tune=False) as b:
            b.run(2)
            upload_noise(b.contexts[1], plans[1], 8)
            b.run(5)
            out.append([x for c in b.contexts for x in levels(c)])
    for u, v in zip(*out):
        assert np.array_equal(u, v)
