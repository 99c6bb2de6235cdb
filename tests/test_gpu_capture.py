"""Steps while the caller captures a stream of its own in the default (global)
mode: the capture goes on and the step is the one it would have been."""
import ctypes

import pytest

import smokesim
from helpers import assert_bitwise_equal, gpu_for, oracle_for
from smokesim import scenes

pytestmark = pytest.mark.gpu


def captured_step(g, dt):
    hip = ctypes.CDLL("libamdhip64.so")
    st, graph = ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(st), 1) == 0
    assert hip.hipStreamBeginCapture(st, 0) == 0
    g.step(dt, readback=False)
    assert hip.hipStreamEndCapture(st, ctypes.byref(graph)) == 0
    assert hip.hipGraphDestroy(graph) == 0 and hip.hipStreamDestroy(st) == 0


@pytest.mark.parametrize("pressure_first", [False, True])
def test_first_reference_step_during_a_capture(pressure_first):
    sc = scenes.test_scene((30, 24, 20), seed=37, projection=smokesim.PROJ_REFERENCE, iterations=6)
    g, o = gpu_for(sc), oracle_for(sc, 32)
    if pressure_first:  # the half-sweeps then allocate a velocity set of their own
        for s in (g, o):
            s.set_params(projection=smokesim.PROJ_JACOBI)
        g.step(sc["dt"], readback=False)
        o.step(sc["dt"])
        for s in (g, o):
            s.set_params(projection=smokesim.PROJ_REFERENCE)
    captured_step(g, sc["dt"])
    g.timing_enable(True)
    g.step(sc["dt"], readback=False)
    assert g.timing_sweeps()[1] < 2 * 6  # several half-sweeps per launch
    o.step(sc["dt"], 2)
    assert_bitwise_equal(g.state(), o.state())
    g.close()
