"""Grids thin in x or y, whose red-black half-sweeps run one per launch where
the marched columns would be mostly empty: bit for bit the FP32 oracle on both
sides of that line, and through a change of the iteration count."""
import numpy as np
import pytest

import smokesim
from helpers import assert_bitwise_equal, gpu_for, oracle_for, random_density
from smokesim import scenes

pytestmark = pytest.mark.gpu


def sweep_launches(g, dt):
    g.timing_enable(True)
    g.timing_reset()
    g.step(dt, readback=False)
    n = g.timing_sweeps()[1]
    g.timing_enable(False)
    return n


@pytest.mark.parametrize("dims,routes", [((3, 4, 2700), {5: True, 1: True, 20: True}),
                                         ((300, 3, 300), {5: True, 1: True, 9: True}),
                                         ((8, 8, 4000), {5: True, 1: True, 9: True}),
                                         ((3, 300, 1400), {5: False, 1: True, 9: False}),
                                         ((40, 2000, 9), {5: True, 20: False, 1: True})], ids=str)
def test_thin_reference_form(dims, routes):
    sc = scenes.test_scene(dims, seed=sum(dims), projection=smokesim.PROJ_REFERENCE, iterations=5, noise=2.0)
    dens = random_density(dims, 5)
    g, o = gpu_for(sc, dens), oracle_for(sc, 32, dens)
    for its, in_place in routes.items():
        for s in (g, o):
            s.set_params(iterations=its)
        n = sweep_launches(g, sc["dt"])
        o.step(sc["dt"])
        assert (n == 2 * its) == in_place, (dims, its, n)
        assert_bitwise_equal(g.state(), o.state(), f"{dims} x{its}")
    g.close()
