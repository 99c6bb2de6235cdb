"""The advection's samples at the ends of the axes: back-traces that stay in the
cell, cross the window of planes a block holds, and are clamped at either end
of every axis, at sizes around the blocks' (64 x 4 cells), against the oracle."""
import numpy as np
import pytest

import smokesim
from helpers import assert_bitwise_equal, gpu_for, oracle_for
from smokesim import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("speed", [0.5, 40.0, 4000.0])
@pytest.mark.parametrize("dims", [(5, 5, 5), (66, 6, 9), (130, 9, 21), (65, 5, 40)])
def test_samples_across_the_grid(dims, speed):
    sc = scenes.test_scene(dims, seed=int(speed) + dims[0], projection=smokesim.PROJ_JACOBI,
                           iterations=3, n_sources=1, n_obstacles=0)
    rng = np.random.default_rng(dims[0])
    g, o = gpu_for(sc), oracle_for(sc, 32)
    for axis in range(3):
        shape = g.get_velocity(axis, 0).shape
        v = rng.uniform(-speed, speed, shape).astype(np.float32)
        for sim in (g, o):
            for half in (0, 1):
                sim.set_velocity(axis, half, v)
    g.step(0.05, readback=False)
    o.step(0.05, 1)
    assert_bitwise_equal(g.state(), o.state(), f"{dims} speed {speed}")
    g.close()
