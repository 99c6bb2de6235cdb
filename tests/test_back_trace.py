"""The density's back-trace in FP32: rounding the double difference of two FP32
values to FP32 gives the FP32 difference, for every cell centre that is an FP32
value and every displacement (the kernels use the FP32 form up to 2^23 cells a
side)."""
import numpy as np
import pytest


@pytest.mark.parametrize("top", [4, 100, 1 << 12, 1 << 23])
def test_fp32_difference_is_the_rounded_double(top):
    rng = np.random.default_rng(top)
    n = 1 << 20
    cell = rng.integers(0, top, n).astype(np.int64)
    cell[:2] = 0, top - 1
    centre = cell.astype(np.float32) + np.float32(0.5)
    assert np.array_equal(centre.astype(np.float64), cell + 0.5)
    exponent = rng.integers(-149, 128, n)
    exponent[: n // 2] = rng.integers(-30, 26, n // 2)  # near the centres' own
    p = np.ldexp(rng.uniform(-2, 2, n), exponent - 1).astype(np.float32)
    p[2:6] = 0.0, -0.0, np.inf, np.nan
    # one unit around the centres' halves, where two roundings could differ
    h = n // 4
    p[h: 2 * h] = np.nextafter(centre[h: 2 * h] * np.float32(0.5), rng.choice([-1e9, 1e9], h)
                               .astype(np.float32))
    with np.errstate(all="ignore"):
        wide = ((cell + 0.5) - p.astype(np.float64)).astype(np.float32)
        assert np.array_equal((centre - p).view(np.uint32)[~np.isnan(p)],
                              wide.view(np.uint32)[~np.isnan(p)])
