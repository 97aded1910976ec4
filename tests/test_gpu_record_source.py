"""Receivers and source in one launch: receivers in the source's cell (one,
several, more than a block) record the stresses ahead of the source, whatever
pieces the steps come in, and the step counter holds through both levels.
FP64 against the oracle, which records in single precision: half a unit of
its last place (2^-24) of the traces' maximum, and 1e-9 for the sums' order."""
import numpy as np
import pytest

import oracle
from opesci import sources
from opesci.backend import Context
from workloads import hetero_model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("at_src,others", [(0, 3), (1, 0), (3, 258), (300, 2), (257, 0)])
@pytest.mark.parametrize("pieces", [(12,), (1, 1, 5, 2, 3)])
def test_receivers_at_the_source(at_src, others, pieces):
    n = sum(pieces)
    g, kw = hetero_model(12, 4, n, double=True, sigma=2.0)
    w = sources.ricker(10.0, g.dt.value, n, t0=4 * g.dt.value) * 50.0
    src = (7, 6, 8)
    rng = np.random.default_rng(5)
    rec = [src] * at_src + [tuple(int(v) for v in rng.integers(2, 14, 3)) for _ in range(others)]
    rec = [rec[i] for i in rng.permutation(len(rec))]
    g.set_source(w, index=src)
    g.set_receivers(index=rec)
    with Context(g.lower()) as ctx:
        ctx.init()
        for k in pieces:
            ctx.run(k)
        tr = ctx.receivers(np.float64)
    ref = oracle.run(src=w, src_idx=src, rec_idx=rec, **kw)['rec']
    assert tr.shape == ref.shape
    assert ref.dtype == np.float32
    assert np.abs(tr - ref).max() <= (2.0 ** -24 + 1e-9) * float(np.abs(ref).max())
