"""Creating a context of a small model: the host work of its boundary program
(hazards of its statements, pieces, groups, one transfer) stays a small part of
a short shot."""
import copy
import time

import pytest

from opesci.backend import Context
from workloads import box_model

pytestmark = pytest.mark.gpu


def seconds(plan):
    t = time.perf_counter()
    ctx = Context(plan)
    t = time.perf_counter() - t
    ctx.close()
    return t


def test_boundary_program_is_cheap_to_create():
    """16^3, 4th order (184 statements): the least of 30 creations with the
    program against the least without its statements.  290 us when every
    rectangle of a statement was compared with all accesses before it, 110 us
    since; the bound lies half way."""
    plan = box_model((16, 16, 16), 4, 10)[0].lower()
    bare = copy.copy(plan)
    bare.stmts = plan.stmts[:0]
    Context(plan).close()
    Context(bare).close()
    times = [(seconds(plan), seconds(bare)) for _ in range(30)]
    assert min(a for a, _ in times) - min(b for _, b in times) < 200e-6
