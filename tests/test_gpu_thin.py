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


@pytest.mark.parametrize("dims,routes", [((51, 4, 6934), {5: True, 1: True, 20: True}),
                                         ((300, 3, 300), {5: True, 1: True, 9: True}),
                                         ((3, 300, 1400), {5: False, 1: False, 9: False}),
                                         ((2449, 40, 9), {5: False, 20: False, 1: False})], ids=str)
@pytest.mark.parametrize("warm", [0, 1])
def test_thin_pressure_form(dims, routes, warm):
    sc = scenes.test_scene(dims, seed=sum(dims), projection=smokesim.PROJ_RBSOR, iterations=5, noise=2.0)
    sc["params"]["warm_start"] = warm
    dens = random_density(dims, 6)
    g, o = gpu_for(sc, dens), oracle_for(sc, 32, dens)
    for its, in_place in routes.items():
        for s in (g, o):
            s.set_params(iterations=its)
        n = sweep_launches(g, sc["dt"])
        o.step(sc["dt"])
        assert (n == 2 * its) == in_place, (dims, its, n)
        assert_bitwise_equal(g.state(), o.state(), f"{dims} x{its}")
        assert np.array_equal(g.get_pressure().view(np.uint32),
                              o.get_pressure().astype(np.float32).view(np.uint32))
    g.close()


# k_ref_pressure_march: 16-pair columns up to 1.5 million cells (test_gpu_redblack.py
# has those), then 32-pair ones with 4 or 6 half-sweeps per launch by their steps:
# 160x142x122 and 158x199x261 with 4 (columns cut in x and y), 241x200x150 with 6.
@pytest.mark.parametrize("dims", [(160, 142, 122), (158, 199, 261)], ids=str)
@pytest.mark.parametrize("iterations,warm", [(1, 0), (2, 1), (7, 1), (13, 0)])
def test_wide_columns_of_four_half_sweeps(dims, iterations, warm):
    sc = scenes.test_scene(dims, seed=iterations, projection=smokesim.PROJ_RBSOR, iterations=iterations,
                           noise=2.0, n_obstacles=2)
    sc["params"]["warm_start"] = warm
    g, o = gpu_for(sc), oracle_for(sc, 32)
    assert sweep_launches(g, sc["dt"]) == -(-2 * iterations // 4)
    g.step(sc["dt"], readback=False)
    o.step(sc["dt"], 2)
    assert_bitwise_equal(g.state(), o.state(), f"{dims} x{iterations}")
    assert np.array_equal(g.get_pressure().view(np.uint32),
                          o.get_pressure().astype(np.float32).view(np.uint32))
    g.close()
