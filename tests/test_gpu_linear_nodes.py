"""Grids whose rows do not fill the bulk kernel's tiles: workgroups take
consecutive nodes, so a wave may start and end anywhere in a row, and hold the
end of a row, of a plane or of the grid.  Moving-lid boxes at row lengths
around the wave and workgroup sizes, every storage-independent path (A/B, AA,
fast and 64-bit-address variants, a layout other than the default): every
population of FP64 runs bit-equal to the oracle."""
import sys

import numpy as np
import pytest

import oracle as orc
from hippolbm_amd import deck as dk
from hippolbm_amd.engine import W, Simulation

pytestmark = pytest.mark.gpu


def deck(n, periodic):
    return dk.loads_msp(f"""
do_domain:
  - domain:
     bounds: [[0,0,0],[{n[0] - 1},{n[1] - 1},{n[2] - 1}]]
     cell_dims: [{n[0] - 1},{n[1] - 1},{n[2] - 1}]
     periodic: [{str(periodic).lower()}, {str(periodic).lower()}, false]
set_lbm_parameters:
  - lbm_parameters:
     tau: 0.8
     nuth: 0.1
pre_stream_bcs:
  - pre_bounce_back
  - cavity_z_l:
     U: [0.05, 0.01, 0]
post_stream_bcs:
  - post_bounce_back
""", "linear_nodes")


# rows of 2..3 nodes (many rows per wave), 63 / 65 (one row end in nearly every
# wave), 64 x 2 planes, 127 / 129 / 193 / 257 (around the tile and workgroup)
SIZES = [(2, 3, 2), (3, 2, 50), (7, 9, 5), (63, 2, 3), (65, 3, 2), (64, 3, 3), (127, 5, 3), (129, 2, 4), (193, 3, 3),
         (257, 2, 2)]


@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("how", ["ab", "aa", "wide", "yzx"])
def test_rows_that_do_not_fill_tiles(n, how):
    print("linear nodes", n, how, flush=True)
    sys.stdout.flush()
    d = deck(n, periodic=how in ("ab", "aa"))
    rng = np.random.default_rng(3)
    rho = 1.0 + 1e-3 * rng.uniform(-1, 1, (n[2], n[1], n[0]))
    f0 = W.reshape(19, 1, 1, 1) * rho
    ref = orc.OracleRun(d, init_f=f0)
    sim = Simulation(d, storage="f64", init_f=f0, pattern="aa" if how == "aa" else "ab")
    if how == "wide":
        sim.dom.set_launch(variant=1)
    if how == "yzx":
        sim.dom.set_layout((1, 2, 0))
    for steps in (1, 4):
        ref.step(steps)
        sim.run(steps)
        assert np.array_equal(sim.dom.get_f(), ref.o.node_f())
    sim.dom.close()


# the last four: under 2 % of the tiles' lanes without a node, taken for rows that are not whole cache lines
@pytest.mark.parametrize("n", SIZES + [(127, 4, 3), (126, 8, 2), (255, 4, 2), (510, 2, 3)],
                         ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("how", ["ab", "aa", "wide", "yzx"])
def test_consecutive_nodes_at_any_size(n, how, monkeypatch):
    """HLBM_LINEAR=2: also below the sizes from which the rule takes them."""
    monkeypatch.setenv("HLBM_LINEAR", "2")
    test_rows_that_do_not_fill_tiles(n, how)


@pytest.mark.parametrize("n", [(47, 48, 44), (47, 48, 45), (63, 74, 75), (63, 75, 76)], ids=lambda n: "x".join(map(str, n)))
def test_the_sizes_from_which_nodes_are_consecutive(n):
    test_rows_that_do_not_fill_tiles(n, "ab")
