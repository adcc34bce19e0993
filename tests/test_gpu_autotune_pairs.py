"""The autotuner's choice between single steps and two steps per pass: whichever
it takes, now or from its cache, the run continues bit for bit, and a launch
shape set by hand is free of an earlier choice."""
import numpy as np
import pytest

from hippolbm_amd.engine import Domain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("storage", ["f64", "f32", "f16"])
def test_tuned_domain_continues_bit_for_bit(storage, monkeypatch):
    n = (128, 65, 64)
    rng = np.random.default_rng(5)
    f0 = (1.0 / 19) * (1.0 + 1e-2 * rng.uniform(-1, 1, (19, n[2], n[1], n[0])))
    out = []
    for pairs, tune in ((0, False), (2, True), (2, True)):  # the second tuning comes from the cache
        monkeypatch.setenv("HLBM_PAIRS", str(pairs))
        dom = Domain(n, (True, True, False), 0.8, (0.0, 0.0, 0.0), storage=storage, collision="bgk", dx=1.0)
        dom.set_bcs([("pre_stream_bcs", "pre_bounce_back", {}), ("post_stream_bcs", "post_bounce_back", {})])
        dom.init_obst()
        dom.set_f(f0)
        dom.step(3)
        if tune:
            dom.autotune(reps=1)
            assert dom.steps_per_pass in (1, 2)
        else:
            assert dom.steps_per_pass == 1
        dom.step(4)
        out.append(dom.get_f())
        if tune:
            dom.set_launch()
            assert dom.steps_per_pass == 2
            dom.set_launch(variant=1)
            assert dom.steps_per_pass == 1
        dom.close()
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])
