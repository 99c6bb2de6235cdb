"""The red-black projections run several half-sweeps per launch on boxes of
the grid: bit for bit the FP32 oracle at the boxes' edges and remainders, for
half-sweep counts that do and do not fill the launches."""
import numpy as np
import pytest

import smokesim
from helpers import assert_bitwise_equal, gpu_for, oracle_for, random_density
from smokesim import scenes

pytestmark = pytest.mark.gpu

# One box, full and cut boxes, then columns (more than 256 boxes) whole and cut
# in x, y and z, and the largest with 6 half-sweeps per launch (5: test_gpu_full_size).
DIMS = [(3, 3, 3), (4, 11, 10), (24, 10, 10), (25, 11, 21), (47, 20, 9), (49, 31, 33), (97, 40, 12),
        (56, 96, 120), (113, 75, 74), (3, 640, 90), (241, 200, 150)]


def scene(dims, projection, iterations, **params):
    sc = scenes.test_scene(dims, seed=sum(dims) + iterations, projection=projection,
                           iterations=iterations, noise=2.0, n_obstacles=2)
    sc["params"].update(params)
    return sc


@pytest.mark.parametrize("dims", DIMS, ids=str)
@pytest.mark.parametrize("iterations", [1, 2, 4, 5, 13])
def test_reference_form(dims, iterations):
    sc = scene(dims, smokesim.PROJ_REFERENCE, iterations)
    dens = random_density(dims, 3)
    g, o = gpu_for(sc, dens), oracle_for(sc, 32, dens)
    for k in range(3):
        g.step(sc["dt"], readback=False)
        o.step(sc["dt"])
        assert_bitwise_equal(g.state(), o.state(), f"{dims} x{iterations} step {k}")
    g.close()


@pytest.mark.parametrize("dims", DIMS, ids=str)
@pytest.mark.parametrize("iterations,warm", [(1, 0), (2, 1), (3, 1), (13, 0)])
def test_pressure_form(dims, iterations, warm):
    sc = scene(dims, smokesim.PROJ_RBSOR, iterations, warm_start=warm)
    dens = random_density(dims, 4)
    g, o = gpu_for(sc, dens), oracle_for(sc, 32, dens)
    for k in range(3):
        if k == 2:  # cells that become solid lose their pressure
            for s in (g, o):
                s.move_object(0, dims[0] / 2, dims[1] / 2, dims[2] / 2)
        g.step(sc["dt"], readback=False)
        o.step(sc["dt"])
        assert_bitwise_equal(g.state(), o.state(), f"{dims} x{iterations} step {k}")
        assert np.array_equal(g.get_pressure().view(np.uint32),
                              o.get_pressure().astype(np.float32).view(np.uint32))
    g.close()


def test_reference_form_keeps_non_finite_faces():
    # An Inf face spreads as Inf and NaN exactly where the oracle's does.
    sc = scene((31, 25, 27), smokesim.PROJ_REFERENCE, 3)
    sc["velocity"][0][9, 8, 7] = np.inf
    g, o = gpu_for(sc), oracle_for(sc, 32)
    for stage in range(3):
        g.run_stage(stage, sc["dt"])
        o.stage(stage, sc["dt"])
    for k in range(3):
        a, b = g.get_velocity(k, 0), o.get_velocity(k, 0).astype(np.float32)
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.isnan(a).any()
        ok = ~np.isnan(a)
        assert np.array_equal(a[ok].view(np.uint32), b[ok].view(np.uint32))
    g.close()
