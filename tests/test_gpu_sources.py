"""All sources are filled by one launch over their bounding boxes: many sources,
overlapping, cut by the walls, outside the grid and empty, bit for bit the
oracle's, in FP32 and in 16-bit storage."""
import numpy as np
import pytest

import smokesim
from helpers import oracle_for
from smokesim import scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [0, 1, 7, 64])
@pytest.mark.parametrize("storage", [smokesim.STORAGE_FP32, smokesim.STORAGE_FP16])
def test_sources(count, storage):
    dims = (37, 21, 30)
    rng = np.random.default_rng(count)
    sc = scenes.test_scene(dims, seed=5, projection=smokesim.PROJ_JACOBI, n_sources=0)
    sc["sources"] = [tuple(np.float32(v) for v in (rng.uniform(-9, 46), rng.uniform(-9, 30),
                                                   rng.uniform(-9, 39), rng.uniform(0.0, 8.0)))
                     for _ in range(count)]
    g = smokesim.Simulation(*dims, storage=storage)
    scenes.apply(g, sc)
    o = oracle_for(sc, 32)
    g.run_stage(smokesim.STAGE_SCENE, sc["dt"])
    o.stage(0, sc["dt"])
    for half in (0, 1):
        assert np.array_equal(g.get_density(half), o.get_density(half).astype(np.float32))
    g.close()
