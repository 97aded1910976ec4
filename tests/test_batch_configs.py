"""The autotuner times no launch shape twice and leaves none of CONFIGS' out."""
import itertools

import pytest

import sweepshape
from opesci.batch import CONFIGS, distinct


class Plan(object):
    def __init__(self, dims, order):
        self.dims, self.order = dims, order


@pytest.fixture(scope="module")
def shape(tmp_path_factory):
    return sweepshape.build(tmp_path_factory.mktemp("shape"))


@pytest.mark.parametrize("order", [2, 4, 8])
def test_configs_are_the_launch_shapes(shape, order):
    for nx, ny, nz in itertools.product((7, 20, 40), (5, 8, 13, 33, 100), (2, 20, 33, 56, 57, 64, 72, 73, 80, 129, 256)):
        plan = Plan((nx + order, ny + order, nz + order), order)

        def launch(cfg):
            # asked-for chunks only: the modelled one (0) is a choice of its own
            s = shape(plan.dims, order // 2, (0, cfg[1], cfg[2] or 1))
            return cfg[0], s['rows'], s['ntz'], s['threads'], s['xc'] if cfg[2] else 0
        kept = distinct(plan)
        assert len({launch(c) for c in kept}) == len(kept), (plan.dims, kept)
        assert {launch(c) for c in kept} == {launch(c) for c in CONFIGS}, (plan.dims, kept)
        assert kept[0] == (0, 0, 0)


def test_tuner_compares_whole_sweeps():
    """every configuration does the z faces where the default does"""
    assert all(c[0] == 0 for c in CONFIGS)
