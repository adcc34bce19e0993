"""Retirement in several batches used in turn: solves of more than 2^18 nodes,
whose statistics fill the whole reduction scratch, among small ones, with
obstacles, both collisions and graph chunks.  What one batch's retirement writes
stays in its own scratch: every solve of every batch gives the fields and the
statistics of the same solve in a batch of its own."""
import numpy as np
import pytest

from hippolbm_amd import batch as bt
from hippolbm_amd.batch import Batch, Solve

pytestmark = pytest.mark.gpu


def solves(seed):
    """Twelve solves, four of each kind: sizes either side of 2^18 nodes, and odd ones."""
    rng = np.random.default_rng(seed)
    sizes = [(64, 64, 64), (67, 66, 61), (31, 31, 31), (65, 33, 20)]
    out = []
    for k in range(12):
        n = sizes[(k + seed) % 4]
        steps = 9 + 4 * ((k + seed) % 4)
        if k % 3 == 0:
            out.append(Solve(nodes=n, steps=steps, tau=0.8, cavity_zl=(float(rng.uniform(0.01, 0.1)), 0.0, 0.0)))
        elif k % 3 == 1:
            out.append(Solve(nodes=n, steps=steps, tau=0.7, periodic=(True, True, False), fext=(1e-5, 0.0, 0.0),
                             collision="mrt"))
        else:
            balls = [{"kind": "ball", "center": tuple(float(rng.uniform(6, m - 7)) for m in n), "radius": 3.0}
                     for _ in range(3)]
            out.append(Solve(nodes=n, steps=steps, tau=0.7, fext=(0.0, 2e-5, 0.0), obstacles=balls,
                             collision="mrt" if k % 2 else "bgk"))
    return out


def collect(b, ids, done):
    for sid in ids:
        if sid not in done and b.state(sid)[0] == bt.DONE:
            stats = b.stats(sid)
            rho, u, _ = b.result(sid)
            done[sid] = (np.array(stats), rho, u)


def test_batches_in_turn_keep_to_their_own_memory():
    work = [solves(seed) for seed in (0, 1, 2)]
    batches = [Batch(storage="f32", budget_bytes=128 << 20, chunk_steps=8) for _ in work]
    ids = [[b.submit(s) for s in w] for b, w in zip(batches, work)]
    done = [{} for _ in work]
    for turn in range(200):
        for b, i, d in zip(batches, ids, done):
            if len(d) < len(i):
                b.run()
                collect(b, i, d)
        if turn % 20 == 0:
            print("turn", turn, [len(d) for d in done], flush=True)
        if all(len(d) == len(i) for d, i in zip(done, ids)):
            break
    for b, i, d in zip(batches, ids, done):
        assert len(d) == len(i)
        b.close()
    alone = Batch(storage="f32", budget_bytes=128 << 20, chunk_steps=8)
    for w, i, d in zip(work, ids, done):
        for s, sid in zip(w, i):
            one, a = {}, alone.submit(s)
            for _ in range(200):
                alone.run()
                collect(alone, [a], one)
                if one:
                    break
            for x, y in zip(d[sid], one[a]):
                assert np.array_equal(x, y)
            rho, u = d[sid][1], d[sid][2]
            # tree and pairwise sums of 3e5 positive terms: some tens of 2^-53 apart
            assert d[sid][0][0] == pytest.approx(rho.sum(), rel=1e-12)
            assert d[sid][0][2] == pytest.approx(np.sqrt((u * u).sum(axis=0)).max(), rel=1e-12)
    alone.close()
