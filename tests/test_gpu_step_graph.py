"""Step graphs beside live steps.  A graph of an even number of steps reads and
writes the buffers it was captured with, and so does every live call of an even
number of steps: replays and such calls may follow each other in any order.  The
two-step kernel, which leaves its result in the other buffer, stays out of a
domain whose steps were captured."""
import ctypes

import numpy as np
import pytest

import oracle as orc
from hippolbm_amd import hip
from hippolbm_amd.engine import W, Simulation

from test_gpu_step_pairs import deck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f64", "f32"])
@pytest.mark.parametrize("captured", [2, 4])
def test_replays_between_live_steps(storage, captured, monkeypatch):
    print("step graph", storage, captured, flush=True)
    n = (70, 30, 20)
    d = deck(n, (1, 0, 0), "bgk", 1e-4)
    f0 = W.reshape(19, 1, 1, 1) * (1.0 + 1e-2 * np.random.default_rng(6).uniform(-1, 1, (19, n[2], n[1], n[0])))
    monkeypatch.setenv("HLBM_PAIRS", "2")
    sim = Simulation(d, storage=storage, init_f=f0)
    dom = sim.dom
    assert dom.steps_per_pass == 2
    dom.step(3)
    stream, h = hip.Stream(), hip.hip()
    hip.device_synchronize()
    graph, ex = ctypes.c_void_p(), ctypes.c_void_p()
    assert h.hipStreamBeginCapture(stream.s, 2) == 0  # relaxed
    dom.step(captured, stream=stream.handle)
    assert h.hipStreamEndCapture(stream.s, ctypes.byref(graph)) == 0
    assert h.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    assert dom.steps_per_pass == 1
    done, fields = 3, []
    for live in (0, 2, 6, 2, 4):  # live calls between the replays
        if live:
            dom.step(live, write_macro=True, stream=stream.handle)
            done += live
            fields.append((done, dom.get_macro()))
        assert h.hipGraphLaunch(ex, stream.s) == 0
        done += captured
        stream.synchronize()
    got = dom.get_f()
    h.hipGraphExecDestroy(ex)
    h.hipGraphDestroy(graph)
    stream.close()
    dom.close()

    # the same steps without a graph, single ones
    monkeypatch.setenv("HLBM_PAIRS", "0")
    one = Simulation(d, storage=storage, init_f=f0)
    at = 0
    for t, (rho, u) in fields:
        one.dom.step(t - at, write_macro=True)
        at = t
        r, v = one.dom.get_macro()
        assert np.array_equal(rho, r) and np.array_equal(u, v)
    one.dom.step(done - at)
    assert np.array_equal(got, one.dom.get_f())
    one.dom.close()
    if storage == "f64":
        ref = orc.OracleRun(d, init_f=f0)
        ref.step(done)
        assert np.array_equal(got, ref.o.node_f())
