"""A simulation whose Jacobi plan was never set takes one fitted to its grid:
the same bits as a plan that was set, for grids of one and of many columns and
chunks, and get_jacobi_plan still returns the default."""
import numpy as np
import pytest

import smokesim
from helpers import assert_bitwise_equal, gpu_for
from smokesim import scenes

pytestmark = pytest.mark.gpu

DIMS = [(3, 3, 3), (24, 25, 4), (34, 23, 57), (56, 46, 100), (150, 40, 260), (260, 250, 90)]


@pytest.mark.parametrize("dims", DIMS, ids=str)
@pytest.mark.parametrize("projection,iterations", [(smokesim.PROJ_JACOBI, 4), (smokesim.PROJ_JACOBI, 11),
                                                   (smokesim.PROJ_REFINED, 20)])
def test_fitted_plan(dims, projection, iterations):
    sc = scenes.test_scene(dims, seed=sum(dims), projection=projection, iterations=iterations, noise=1.0)
    a, b = gpu_for(sc), gpu_for(sc)
    default = a.get_jacobi_plan()
    b.set_jacobi_plan(**default)
    for _ in range(2):
        a.step(sc["dt"], readback=False)
        b.step(sc["dt"], readback=False)
    assert a.get_jacobi_plan() == default == dict(sweeps_per_launch=4, tile=0, zc=64)
    assert_bitwise_equal(a.state(), b.state(), f"{dims}")
    assert np.array_equal(a.get_pressure().view(np.uint32), b.get_pressure().view(np.uint32))
    a.close()
    b.close()
