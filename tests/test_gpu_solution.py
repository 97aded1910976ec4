"""The analytic-solution point kernels against the plan interpreter for every
way a program can go: several points at once (stack depth to 5), one point at
a time (deeper), and programs that hold POWC, EXP or LOG.

Tolerance: the FP64 contract of the parity tests, 1e-12 of the field maximum
(the programs here are at most 14 operations of a few 2^-53 each)."""
import numpy as np
import pytest

from opesci import exprvm
from opesci.backend import Context
from planvm import PlanVM
from workloads import box_model

pytestmark = pytest.mark.gpu

X, Y, Z = ((exprvm.OP_COORD, (a, 0, 0, 0), 0.0) for a in range(3))
MU = (exprvm.OP_MEDIA, (exprvm.MEDIA_IDS['mu'], 0, 0, 0), 0.0)


def op(o, val=0.0):
    return (o, (0, 0, 0, 0), val)


def nested(depth):
    """a + (b * (c + (... * mu))) over the axes in turn: stack depth `depth`,
    no part of one axis only that a table could hold"""
    axes = [(X, Y, Z)[i % 3] for i in range(depth - 1)]
    return axes + [MU] + [op(exprvm.OP_ADD if i % 2 else exprvm.OP_MUL) for i in range(depth - 1)]


ELEM = [MU, X, op(exprvm.OP_ADD), op(exprvm.OP_LOG), Y, op(exprvm.OP_MUL), op(exprvm.OP_EXP),
        Z, op(exprvm.OP_ADD), op(exprvm.OP_POWC, 1.5)]
PLAIN = [X, MU, op(exprvm.OP_DIV), op(exprvm.OP_SQRT), op(exprvm.OP_SIN), Y, op(exprvm.OP_COS), op(exprvm.OP_SUB)]


@pytest.mark.parametrize("programs", [
    [PLAIN, nested(3), nested(4), nested(5)],
    [PLAIN, nested(5), nested(6), nested(9)],
    [ELEM, PLAIN, nested(5)],
    [nested(7), ELEM],
], ids=['fit', 'deep', 'elem', 'both'])
@pytest.mark.parametrize("sizes", [(3, 5, 7), (9, 6, 258)])
def test_solution_program_forms(programs, sizes):
    g, _ = box_model(sizes, 2, 1, hetero=True, double=True)
    plan = g.lower()
    code, off, ln = [], [], []
    for f in range(9):
        c = programs[f % len(programs)]
        off.append(len(code))
        ln.append(len(c))
        code += c
    plan.sol_code, plan.sol_off, plan.sol_len = exprvm.to_array(code), off, ln
    vm = PlanVM(plan)
    with np.errstate(all='ignore'):
        vm.init()
    with Context(plan) as ctx:
        ctx.init()
        got = [ctx.download(f, 0) for f in range(9)]
    for f in range(9):
        want = vm.F[f, 0]
        assert np.isfinite(want).all() and np.abs(want).max() > 0.0
        assert np.abs(got[f] - want).max() <= 1e-12 * np.abs(want).max(), f
