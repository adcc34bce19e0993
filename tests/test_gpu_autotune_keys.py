"""What the autotuner keeps for later domains of the same size: a choice made
where two steps per pass do not apply (walls, start_iteration boxes, a layout set
by hand, a mode of the environment, captured steps) is not taken by a domain
where they do, and the other way round; the same domain again takes the choice
from the cache, steps per pass included.  On one domain, a choice made while
walls stood does not outlast them."""
import numpy as np
import pytest

from hippolbm_amd import hip
from hippolbm_amd.engine import Domain

pytestmark = pytest.mark.gpu

BCS = [("pre_stream_bcs", "pre_bounce_back", {}), ("post_stream_bcs", "post_bounce_back", {})]


def make(n, bcs=BCS):
    dom = Domain(n, (True, True, False), 0.8, (0.0, 0.0, 0.0), storage="f32", collision="bgk", dx=1.0)
    dom.set_bcs(bcs)
    dom.init_obst()
    dom.set_distribution(1.0)
    return dom


def with_walls(n, monkeypatch):
    dom = make(n)
    dom.add_obstacles([{"kind": "ball", "center": (10.0, 10.0, 10.0), "radius": 3.0}])  # no wall_bounce_back
    return dom


def with_box(n, monkeypatch):
    return make(n, [("start_iteration", "set_distribution", {"value": 1.0, "bounds": ((0.0, 0.0, 0.0), (3.0, 3.0, 3.0))})] + BCS)


def with_layout(n, monkeypatch):
    dom = make(n)
    dom.set_layout((1, 2, 0))
    return dom


def with_pairs_off(n, monkeypatch):
    monkeypatch.setenv("HLBM_PAIRS", "0")
    dom = make(n)
    monkeypatch.setenv("HLBM_PAIRS", "2")
    return dom


def with_wide(n, monkeypatch):
    monkeypatch.setenv("HLBM_FORCE_WIDE", "1")
    dom = make(n)
    monkeypatch.delenv("HLBM_FORCE_WIDE")
    return dom


def with_captured_steps(n, monkeypatch):
    import ctypes
    dom = make(n)
    dom.step(1)
    stream, graph = hip.Stream(), ctypes.c_void_p()
    hip.device_synchronize()
    assert hip.hip().hipStreamBeginCapture(stream.s, 2) == 0
    dom.step(2, stream=stream.handle)
    assert hip.hip().hipStreamEndCapture(stream.s, ctypes.byref(graph)) == 0
    hip.hip().hipGraphDestroy(graph)
    stream.close()
    return dom


# a size of its own for every case: the cache lives as long as the process
@pytest.mark.parametrize("other,n", [(with_walls, (66, 28, 26)), (with_box, (66, 28, 27)), (with_layout, (66, 28, 28)),
                                     (with_pairs_off, (66, 28, 29)), (with_wide, (66, 28, 30)),
                                     (with_captured_steps, (66, 28, 31))], ids=lambda v: getattr(v, "__name__", None))
@pytest.mark.parametrize("first", ["other", "plain"])
def test_choices_are_kept_apart(other, n, first, monkeypatch):
    n = n if first == "other" else (n[0] + 1, n[1], n[2])
    print("autotune key", other.__name__, n, first, flush=True)
    monkeypatch.setenv("HLBM_PAIRS", "2")
    a, b = other(n, monkeypatch), make(n)
    assert (a.steps_per_pass, b.steps_per_pass) == (1, 2)
    info = {}
    for dom in (a, b) if first == "other" else (b, a):
        info[dom] = dom.autotune(reps=1)
        assert info[dom]["candidates"] > 0  # measured, not taken from the other's entry
    assert a.steps_per_pass == 1
    assert b.get_layout() == (0, 1, 2)
    c = make(n)
    again = c.autotune(reps=1)
    assert again["candidates"] == 0 and again["block"] == info[b]["block"] and again["variant"] == info[b]["variant"]
    assert c.steps_per_pass == b.steps_per_pass
    for dom in (a, b, c):
        dom.step(7)
    assert np.array_equal(b.get_f(), c.get_f())
    for dom in (a, b, c):
        dom.close()


def test_a_choice_made_with_walls_does_not_outlast_them(monkeypatch):
    """Whatever shape the walls' steps were tuned to, the 64-bit variant included,
    the domain makes two steps per pass once the walls are gone."""
    monkeypatch.setenv("HLBM_PAIRS", "2")
    n = (70, 31, 27)
    f0 = (1.0 / 19) * (1.0 + 1e-2 * np.random.default_rng(8).uniform(-1, 1, (19, n[2], n[1], n[0])))
    out = []
    for tuned in (True, False):
        dom = make(n)
        dom.add_obstacles([{"kind": "ball", "center": (10.0, 10.0, 10.0), "radius": 3.0}])
        dom.set_f(f0)
        if tuned:
            dom.autotune(reps=1)
        assert dom.steps_per_pass == 1
        dom.step(3)
        dom.init_obst()
        assert dom.steps_per_pass == 2
        dom.step(6)
        out.append(dom.get_f())
        dom.close()
    assert np.array_equal(*out)


def test_a_shape_set_by_hand_holds(monkeypatch):
    """Variant 1 asked for by hand stays one step per pass, through a change of the
    collision too; variant 0 leaves the rule."""
    monkeypatch.setenv("HLBM_PAIRS", "2")
    dom = make((66, 20, 18))
    dom.set_launch(variant=1)
    assert dom.steps_per_pass == 1
    dom.set_collision("mrt")
    assert dom.steps_per_pass == 1
    dom.set_launch(variant=0)
    assert dom.steps_per_pass == 2
    dom.close()
