"""Two handles at once from two threads, as the C ABI allows: kernels whose workgroups wait for each other
(the level walk, the batched launch's teams) side by side on the device.  Every result is the one that the
same call gives alone, and none runs into a deadline."""
import threading

import numpy as np
import pytest

from batchlayoutcode_amd import graphs

pytestmark = pytest.mark.gpu


def _both(jobs, rounds):
    """Runs the jobs alone, then `rounds` times each at once; returns both sides' results."""
    alone = [job() for job in jobs]
    start = threading.Barrier(len(jobs))
    got, errors = [[] for _ in jobs], []

    def work(k):
        try:
            start.wait(30)
            for _ in range(rounds):
                got[k].append(jobs[k]())
        except BaseException as e:  # noqa: BLE001 (shown by the caller)
            errors.append(e)

    ts = [threading.Thread(target=work, args=(k,)) for k in range(len(jobs))]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors
    return alone, got


def test_two_level_walks_at_once(bl):
    made = [graphs.csr_from_edges(*graphs.rgg(120_000, seed=5)), graphs.csr_from_edges(*graphs.rmat(17, 8, seed=2)[:2])]
    print("[case] two level walks at once", [len(rp) - 1 for rp, _ in made], flush=True)
    handles = [bl.Graph(rp, ci) for rp, ci in made]
    xs = [np.random.default_rng(k).random((len(rp) - 1, 2)) for k, (rp, _) in enumerate(made)]

    def job(k):
        return lambda: handles[k].run(xs[k], algo=4, iters=10, batch=(256, 1024)[k], bht=1.2)

    alone, got = _both([job(0), job(1)], 12)
    for k in (0, 1):
        for xy, st in got[k]:
            assert np.array_equal(xy, alone[k][0]) and st.energy == alone[k][1].energy
        handles[k].close()


def test_two_batched_launches_at_once(bl):
    sets = []
    for seed in (1, 2):
        rng = np.random.default_rng(seed)
        gs, xs = [], []
        for n in rng.integers(200, 8192, 60):
            e = rng.integers(0, n, (4 * n, 2))
            gs.append(graphs.csr_from_edges(int(n), e[e[:, 0] != e[:, 1]]))
            xs.append(rng.random((int(n), 2)))
        sets.append((gs, xs))
    print("[case] two batched launches at once", flush=True)
    alone, got = _both([lambda s=s: bl.run_batched(*s, algo=2, iters=10, batch=128) for s in sets], 4)
    for k in (0, 1):
        for out, en, _, _ in got[k]:
            assert all(np.array_equal(a, b) for a, b in zip(out, alone[k][0])) and np.array_equal(en, alone[k][1])
