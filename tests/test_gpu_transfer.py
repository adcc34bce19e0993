"""Populations, density and velocity between the device and host arrays, at
sizes around the ones from which they go through the pinned ring (rearranged
planes 4 MiB in all, others 12 MiB to the host and 32 MiB to the device): a ring
not filled once, rows and planes that straddle chunks, more chunks than slots,
the larger slots from 64 MiB on, a device layout other than the host's, the
reference layout with its ghost layers, each storage.

Exact: the host form of a stored population is a fixed sequence of IEEE
operations, restated here in numpy."""
import numpy as np
import pytest

from hippolbm_amd import _lib
from hippolbm_amd.engine import CX, CY, CZ, W, Domain

pytestmark = pytest.mark.gpu


def stored(f, storage):
    """f as it comes back from the storage type (BGK: shifted by w)."""
    if storage == "f64":
        return f
    w = W.reshape(19, 1, 1, 1)
    g = (f - w).astype(np.float32)
    if storage == "f16":
        g = (g * np.float32(8192)).astype(np.float16).astype(np.float32) * np.float32(2.0 ** -13)
    elif storage == "bf16":
        b = g.view(np.uint32)
        g = ((b + np.uint32(0x7FFF) + ((b >> np.uint32(16)) & np.uint32(1))) & np.uint32(0xFFFF0000)).view(np.float32)
    return g.astype(np.float64) + w


# 30 x 30 x 30 and 31 x 30 x 30, 43^3 and 44^3: either side of the populations' 4 and 12 MiB; 64 x 64 x 31 and
# 64 x 64 x 32: of the fields' 4 MiB; 59^3 and 61^3: of 32 MiB to the device; odd rows; 64 MiB and more
SIZES = [(30, 30, 30), (31, 30, 30), (43, 43, 43), (44, 44, 44), (64, 64, 31), (64, 64, 32), (59, 59, 59), (61, 61, 61),
         (131, 67, 61), (129, 130, 131)]


@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("storage", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("order", [(0, 1, 2), (1, 2, 0)], ids=["xyz", "yzx"])
def test_host_arrays_round_trip(n, storage, order):
    print("transfer", n, storage, order, flush=True)
    rng = np.random.default_rng(5)
    shape = (n[2], n[1], n[0])
    f = W.reshape(19, 1, 1, 1) * (1.0 + 0.02 * rng.uniform(-1, 1, (19,) + shape))
    want = stored(f, storage)
    dom = Domain(n, (True, False, False), 0.8, storage=storage)
    dom.set_layout(order)
    dom.init_obst()
    dom.set_f(f)
    assert np.array_equal(dom.get_f(), want)
    # the reference layout: Real nodes inside two ghost layers, periodic x filled, the rest left alone
    ref = dom.get_f(_lib.LAYOUT_REF, out=np.full((19,) + tuple(v + 4 for v in shape), 7.0))
    assert np.array_equal(ref[:, 2:-2, 2:-2, 2:-2], want)
    assert np.array_equal(ref[:, 2:-2, 2:-2, :2], want[..., -2:])
    assert (ref[:, :2] == 7.0).all() and (ref[:, :, -2:] == 7.0).all()
    if n[0] % 2:
        pad = np.full_like(ref, 3.0)
        pad[:, 2:-2, 2:-2, 2:-2] = f[:, ::-1]
        dom.set_f(pad, _lib.LAYOUT_REF)
        assert np.array_equal(dom.get_f(), stored(f[:, ::-1], storage))
        dom.set_f(f)
    rho, u = dom.macro()
    rho2, u2 = dom.get_macro(_lib.LAYOUT_REF)
    assert np.array_equal(rho2[2:-2, 2:-2, 2:-2], rho) and np.array_equal(u2[:, 2:-2, 2:-2, 2:-2], u)
    if storage == "f64":
        want_rho = np.zeros(shape)
        j = np.zeros((3,) + shape)
        for i in range(19):
            for d, c in enumerate((CX[i], CY[i], CZ[i])):
                if c:
                    j[d] += c * f[i]
            want_rho += f[i]
        assert np.array_equal(rho, want_rho) and np.array_equal(u, j / want_rho)
    dom.close()
