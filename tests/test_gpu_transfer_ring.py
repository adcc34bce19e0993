"""The pinned ring of large host transfers over its life: one that grows with the
first transfer of 64 MiB, one that passes from a destroyed domain to the next
(other sizes, storages and layouts), several at once, each domain on a thread of
its own, and one given back after enough domains without large transfers.  Exact,
like the single transfers; and round trips at the sizes from which populations in
the reference layout take the ring to the host."""
import threading

import numpy as np
import pytest

from hippolbm_amd import _lib
from hippolbm_amd.engine import W, Domain

from test_gpu_transfer import stored
from test_gpu_transfer import test_host_arrays_round_trip as round_trip

pytestmark = pytest.mark.gpu


def populations(n, seed):
    rng = np.random.default_rng(seed)
    return W.reshape(19, 1, 1, 1) * (1.0 + 0.02 * rng.uniform(-1, 1, (19, n[2], n[1], n[0])))


def make(n, storage="f64", order=(0, 1, 2)):
    dom = Domain(n, (True, False, False), 0.8, storage=storage)
    dom.set_layout(order)
    dom.init_obst()
    return dom


def check(dom, n, storage, seed, layout=_lib.LAYOUT_NODES):
    """In and out again, populations, then the density they give."""
    f = populations(n, seed)
    dom.set_f(f)
    want = stored(f, storage)
    got = dom.get_f(layout)
    assert np.array_equal(got if layout == _lib.LAYOUT_NODES else got[:, 2:-2, 2:-2, 2:-2], want)
    if storage == "f64":
        rho = np.zeros(want.shape[1:])
        for i in range(19):
            rho += f[i]
        assert np.array_equal(dom.macro()[0], rho)


# 19 x 34^3 and 35^3 doubles: either side of 6 MiB
@pytest.mark.parametrize("n", [(34, 34, 34), (35, 35, 35)], ids=lambda n: "x".join(map(str, n)))
@pytest.mark.parametrize("storage", ["f64", "f32", "f16", "bf16"])
@pytest.mark.parametrize("order", [(0, 1, 2), (1, 2, 0)], ids=["xyz", "yzx"])
def test_sizes_from_which_the_reference_layout_takes_the_ring(n, storage, order):
    round_trip(n, storage, order)


def test_a_ring_grows_and_serves_small_transfers_again():
    """Fields of 12.5 MiB, populations of 8.6 x that (the second block), fields again."""
    n = (74, 74, 75)
    dom = make(n)
    for seed in (1, 2):
        f = populations(n, seed)
        dom.set_f(f)
        rho, u = dom.macro()
        assert np.array_equal(dom.get_f(), f)
        again = dom.get_macro()
        assert np.array_equal(rho, again[0]) and np.array_equal(u, again[1])
        rho_ref = dom.get_macro(_lib.LAYOUT_REF)[0]
        assert np.array_equal(rho_ref[2:-2, 2:-2, 2:-2], rho)
    dom.close()


def test_a_ring_passes_from_domain_to_domain():
    cases = [((96, 80, 64), "f64", (0, 1, 2)), ((61, 60, 59), "f32", (0, 1, 2)), ((40, 41, 43), "f16", (1, 2, 0)),
             ((97, 83, 65), "bf16", (0, 1, 2)), ((52, 52, 52), "f64", (1, 2, 0)), ((48, 49, 50), "f64", (0, 1, 2))]
    for seed, (n, storage, order) in enumerate(cases):
        print("ring", n, storage, order, flush=True)
        dom = make(n, storage, order)
        check(dom, n, storage, seed)
        check(dom, n, storage, seed + 50, _lib.LAYOUT_REF)
        dom.close()


def test_idle_domains_give_the_ring_back():
    for seed in range(2):
        dom = make((52, 52, 52))
        check(dom, (52, 52, 52), "f64", seed)
        dom.close()
        for _ in range(10):  # more than the ring waits for
            make((8, 8, 8)).close()


def test_domains_on_threads_of_their_own():
    n = [(61, 60, 59), (52, 53, 54), (75, 74, 73)]
    failed = []

    def work(k):
        try:
            for turn in range(3):
                dom = make(n[k])
                check(dom, n[k], "f64", 10 * k + turn)
                dom.close()
        except BaseException as e:  # reported by the test's own thread
            failed.append((k, repr(e)[:500]))

    threads = [threading.Thread(target=work, args=(k,)) for k in range(len(n))]
    for t in threads:
        t.start()
    for t in threads:
        t.join(60)
    assert not failed and not any(t.is_alive() for t in threads)
