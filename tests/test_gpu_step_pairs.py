"""Two steps per pass (pair_kernel) against single steps and the oracle.

HLBM_PAIRS=2 takes the two-step kernel at every size, HLBM_PAIRS=0 never.  The
node's arithmetic is the same code, so every population must be equal bit for
bit: FP64 against the oracle, the reduced storages (16-bit ones, BGK, rounding
stochastically in between) against single steps.  Sizes around the tile
(64 columns, 13 rows) and the segment, with rings that wrap onto the tile
itself, faces on every axis and their edges and corners (the moving wall
included), odd and even step counts, rho and u of the last step."""
import ctypes

import numpy as np
import pytest

import oracle as orc
from hippolbm_amd import deck as dk
from hippolbm_amd.engine import W, Simulation

pytestmark = pytest.mark.gpu

# one tile and less; exactly one, one more; 12, 13 and 26 rows; several segments
SIZES = [(2, 2, 2), (5, 3, 4), (64, 9, 6), (65, 10, 5), (63, 12, 7), (128, 13, 3), (130, 26, 9), (20, 7, 64), (17, 5, 66),
         (9, 11, 130)]


def deck(n, periodic, collision, force):
    flags = ", ".join("true" if v else "false" for v in periodic)
    lid = "  - cavity_z_l:\n     U: [0.05, 0.01, 0]\n  - cavity_z_0:\n     U: [-0.02, 0.03, 0]\n" if not periodic[2] else ""
    return dk.loads_msp(f"""
do_domain:
  - domain:
     bounds: [[0,0,0],[{n[0] - 1},{n[1] - 1},{n[2] - 1}]]
     cell_dims: [{n[0] - 1},{n[1] - 1},{n[2] - 1}]
     periodic: [{flags}]
set_lbm_parameters:
  - lbm_parameters:
     tau: 0.7
     nuth: {0.2 / 3!r}
     Fext: [{force!r}, 0, {force!r}]
collision: {collision}
pre_stream_bcs:
  - pre_bounce_back
{lid}post_stream_bcs:
  - post_bounce_back
""", "step_pairs")


def start(d, n, storage, monkeypatch, pairs, f0):
    monkeypatch.setenv("HLBM_PAIRS", str(pairs))
    return Simulation(d, storage=storage, init_f=f0)


@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("periodic", [(1, 1, 0), (0, 0, 0), (1, 0, 1), (1, 1, 1), (0, 1, 0)],
                         ids=lambda p: "p" + "".join(map(str, p)))
@pytest.mark.parametrize("collision", ["bgk", "mrt"])
def test_pairs_equal_single_steps(n, periodic, collision, monkeypatch):
    print("pairs", n, periodic, collision, flush=True)
    d = deck(n, periodic, collision, 1e-4 if collision == "bgk" else 0.0)
    rng = np.random.default_rng(1)
    f0 = W.reshape(19, 1, 1, 1) * (1.0 + 1e-2 * rng.uniform(-1, 1, (19, n[2], n[1], n[0])))
    ref = orc.OracleRun(d, init_f=f0)
    sim = start(d, n, "f64", monkeypatch, 2, f0)
    for steps in (3, 4):  # after the collide-only step: one pair; then two pairs, or one step and a pair
        ref.step(steps)
        sim.run(steps)
        assert np.array_equal(sim.dom.get_f(), ref.o.node_f())
    sim.run(6)
    rho, u = sim.dom.get_macro()
    f = sim.dom.get_f()
    sim.dom.close()
    one = start(d, n, "f64", monkeypatch, 0, f0)
    for steps in (3, 4, 6):
        one.run(steps)
        last = one.dom.get_macro()
        one.dom.get_f()
    assert np.array_equal(rho, last[0]) and np.array_equal(u, last[1])
    assert np.array_equal(f, one.dom.get_f())
    one.dom.close()
    for storage in ("f32", "f16", "bf16"):
        runs = []
        for pairs in (2, 0):
            s = start(d, n, storage, monkeypatch, pairs, f0)
            s.run(8)
            runs.append((s.dom.get_f(),) + s.dom.get_macro())
            s.dom.close()
        for a, b in zip(*runs):
            assert np.array_equal(a, b), storage


@pytest.mark.parametrize("n", [(130, 92, 92), (130, 92, 93), (257, 67, 65)], ids=lambda n: "x".join(map(str, n)))
def test_pairs_above_the_cache(n, monkeypatch):
    """FP64 below and above the 320 MiB from which the populations are stored
    with the non-temporal hint: the largest size of the plain stores, the next
    one and a ragged one, equal to single steps bit for bit."""
    print("pairs above the cache", n, flush=True)
    d = deck(n, (1, 0, 0), "bgk", 1e-4)
    f0 = W.reshape(19, 1, 1, 1) * (1.0 + 1e-2 * np.random.default_rng(2).uniform(-1, 1, (19, n[2], n[1], n[0])))
    runs = []
    for pairs in (2, 0):
        sim = start(d, n, "f64", monkeypatch, pairs, f0)
        sim.run(5)
        runs.append(sim.dom.get_f())
        sim.dom.close()
    assert np.array_equal(runs[0], runs[1])


def test_captured_steps_replay(monkeypatch):
    """A captured call of two steps advances by two steps on every replay: it
    holds single steps, which return to the buffer they started from."""
    from hippolbm_amd import hip
    n = (70, 30, 20)
    d = deck(n, (1, 0, 0), "bgk", 1e-4)
    f0 = W.reshape(19, 1, 1, 1) * (1.0 + 1e-2 * np.random.default_rng(6).uniform(-1, 1, (19, n[2], n[1], n[0])))
    sim = start(d, n, "f64", monkeypatch, 2, f0)
    sim.run(3)
    stream, h = hip.Stream(), hip.hip()
    hip.device_synchronize()
    graph, ex = ctypes.c_void_p(), ctypes.c_void_p()
    assert h.hipStreamBeginCapture(stream.s, 2) == 0  # relaxed
    sim.dom.step(2, stream=stream.handle)
    assert h.hipStreamEndCapture(stream.s, ctypes.byref(graph)) == 0
    assert h.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
    for _ in range(3):
        assert h.hipGraphLaunch(ex, stream.s) == 0
        stream.synchronize()
    got = sim.dom.get_f()
    h.hipGraphExecDestroy(ex)
    h.hipGraphDestroy(graph)
    stream.close()
    sim.dom.close()
    ref = orc.OracleRun(d, init_f=f0)
    ref.step(9)
    assert np.array_equal(got, ref.o.node_f())
