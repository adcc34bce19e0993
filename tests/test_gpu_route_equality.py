"""Calls that a rule on sizes takes to another kernel give what the general path
gives, bit for bit, in the forms that the rule accepts beside the plain ones:
consecutive nodes (HLBM_LINEAR=2) against tiles (0) with obstacles, walls next to
a periodic face, open planes, MRT and BGK, every storage, A/B and AA, a layout
other than the default, the 64-bit variant; two steps per pass (HLBM_PAIRS=2)
against single steps (0) for MRT with a body force and for 16-bit storage rounded
to nearest; and the rules' own choices on either side of their lines."""
import numpy as np
import pytest

from hippolbm_amd import deck as dk
from hippolbm_amd.engine import W, Domain, Simulation

from test_gpu_parity import _channel_deck, _porous_deck
from test_gpu_periodic_walls import WALL_AT_FACE
from test_gpu_step_pairs import deck as box_deck

pytestmark = pytest.mark.gpu

DECKS = {
    "channel": lambda: _channel_deck(41, 19, 17, 5, 3, "mrt"),
    "channel_bgk": lambda: _channel_deck(67, 18, 15, 4, 3, "bgk"),
    "spheres": lambda: _porous_deck(37, 21, 19, 5, 7, "bgk"),
    "spheres_mrt": lambda: _porous_deck(65, 20, 18, 5, 9, "mrt"),
    "periodic_wall": lambda: dk.loads_msp(WALL_AT_FACE, "periodic_wall"),
}


def outputs(sim, *runs):
    out = []
    for steps in runs:
        sim.run(steps)
        out += list(sim.dom.get_macro())
        out.append(sim.dom.get_f())
    sim.dom.close()
    return out


@pytest.mark.parametrize("name", DECKS)
@pytest.mark.parametrize("storage", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("how", ["ab", "aa", "yzx", "wide"])
def test_consecutive_nodes_equal_tiles(name, storage, how, monkeypatch):
    print("linear", name, storage, how, flush=True)
    res = []
    for linear in (0, 2):
        monkeypatch.setenv("HLBM_LINEAR", str(linear))
        sim = Simulation(DECKS[name](), storage=storage, pattern="aa" if how == "aa" else "ab")
        if how == "yzx":
            sim.dom.set_layout((1, 2, 0))
        if how == "wide":
            sim.dom.set_launch(variant=1)
        res.append(outputs(sim, 5, 6))
    for a, b in zip(*res):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("n", [(65, 14, 9), (20, 7, 66)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("periodic", [(1, 1, 0), (0, 0, 0), (0, 1, 1)], ids=lambda p: "p" + "".join(map(str, p)))
@pytest.mark.parametrize("storage,collision,rounding", [("f64", "mrt", "stochastic"), ("f32", "mrt", "stochastic"),
                                                        ("f16", "bgk", "nearest"), ("bf16", "bgk", "nearest")])
def test_pairs_equal_single_steps_in_the_other_forms(n, periodic, storage, collision, rounding, monkeypatch):
    print("pairs", n, periodic, storage, collision, rounding, flush=True)
    d = box_deck(n, periodic, collision, 1e-4)
    f0 = W.reshape(19, 1, 1, 1) * (1.0 + 1e-2 * np.random.default_rng(4).uniform(-1, 1, (19, n[2], n[1], n[0])))
    res = []
    for pairs in (0, 2):
        monkeypatch.setenv("HLBM_PAIRS", str(pairs))
        sim = Simulation(d, storage=storage, init_f=f0, rounding=rounding)
        assert sim.dom.steps_per_pass == (2 if pairs else 1)
        res.append(outputs(sim, 5, 6, 3))
    for a, b in zip(*res):
        assert np.array_equal(a, b)


# the rule's fill (the domain's share of the lanes and planes that the launch steps) on either side of its line
@pytest.mark.parametrize("n,storage,passes", [((97, 97, 97), "f64", 2), ((63, 80, 80), "f64", 1), ((64, 64, 64), "f32", 2),
                                              ((48, 48, 48), "f32", 1), ((256, 200, 100), "f16", 2),
                                              ((128, 128, 128), "f16", 1), ((250, 200, 100), "bf16", 1)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_the_rule_for_two_steps_per_pass(n, storage, passes, monkeypatch):
    print("rule", n, storage, flush=True)
    res = []
    for pairs in (None, "0"):
        if pairs is None:
            monkeypatch.delenv("HLBM_PAIRS", raising=False)
        else:
            monkeypatch.setenv("HLBM_PAIRS", pairs)
        dom = Domain(n, (True, False, False), 0.8, (1e-6, 0.0, 0.0), storage=storage)
        dom.set_bcs([("pre_stream_bcs", "pre_bounce_back", {}), ("pre_stream_bcs", "cavity_z_l", {"U": (0.05, 0.01, 0.0)}),
                     ("post_stream_bcs", "post_bounce_back", {})])
        dom.init_obst()
        dom.set_distribution(1.0)
        dom.set_distribution(1.01, ((1, 2, 3), (9, 8, 7)))
        assert dom.steps_per_pass == (passes if pairs is None else 1)
        dom.step(6, write_macro=True)
        res.append(dom.get_macro() + (dom.get_f(),))
        dom.close()
    for a, b in zip(*res):
        assert np.array_equal(a, b)
