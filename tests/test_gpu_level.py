"""The batch walk by dependence levels against the sequential walks it replaces.

Every vertex reads the positions it would read in the sequential walk, so the layouts agree up to
the order of partial sums (1e-10 of the diameter after one iteration, the bar of the other
walks), and bit for bit where the levels keep the lagged walk's sums.
"""
import numpy as np
import pytest

from batchlayoutcode_amd import graphs
from conftest import diameter

pytestmark = pytest.mark.gpu


def _path(n):
    i = np.arange(n - 1)
    return graphs.csr_from_edges(n, np.stack([i, i + 1], 1))


def _star(n, hubs, seed):
    """Late hubs (ids at the end, so all their neighbours are early) over a random graph."""
    rng = np.random.default_rng(seed)
    e = [rng.integers(0, n, size=(2 * n, 2))]
    for k in range(hubs):
        others = rng.choice(n - hubs, 65 + k * (n // (hubs + 1)), replace=False)
        e.append(np.stack([np.full(len(others), n - 1 - k), others], 1))
    e = np.unique(np.sort(np.concatenate(e), 1), axis=0)
    return graphs.csr_from_edges(n, e[e[:, 0] != e[:, 1]])


def _one_way(n, seed):
    """Rows in any order, with duplicates and self-loops, and no edge needing its reverse."""
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 12, n)
    rp = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    return rp, rng.integers(0, n, rp[-1]).astype(np.int32)


def _make(kind):
    if kind == "path":
        return _path(3000)
    if kind == "grid":  # natural order: levels of about a row of the grid, in one workgroup
        return graphs.csr_from_edges(*graphs.grid(70, 900))
    if kind == "widegrid":  # levels of 2100 vertices, more than one workgroup takes
        return graphs.csr_from_edges(*graphs.grid(20, 2100))
    if kind == "rgg":
        return graphs.csr_from_edges(*graphs.rgg(30_000, seed=5))
    if kind == "hubs":
        return _star(12_000, 7, 3)
    if kind == "one_way":
        return _one_way(5000, 4)
    if kind == "edgeless":
        return np.zeros(301, np.int32), np.zeros(0, np.int32)
    return graphs.csr_from_edges(*graphs.rmat(13, 8, seed=2)[:2])


@pytest.mark.parametrize("kind,batch,algo,weighted,prec", [
    ("path", 1, 4, False, 0), ("path", 64, 40, True, 0), ("grid", 64, 4, False, 0), ("grid", 333, 4, True, 2),
    ("widegrid", 100, 4, False, 0), ("rgg", 1000, 40, True, 0), ("rgg", 63, 4, False, 0), ("hubs", 256, 4, False, 0),
    ("hubs", 1000, 4, True, 0), ("one_way", 128, 4, False, 0), ("one_way", 4096, 4, True, 0),
    ("edgeless", 16, 4, False, 0), ("rmat", 100, 40, True, 0), ("rmat", 3000, 4, False, 0)])
def test_levels_match_the_sequential_walk(bl, monkeypatch, kind, batch, algo, weighted, prec):
    rp, ci = _make(kind)
    n = len(rp) - 1
    w = np.random.default_rng(7).uniform(0.5, 2.0, len(ci)).astype(np.float32) if weighted else None
    x0 = np.random.default_rng(8).random((n, 2))
    print(f"[case] levels {kind} batch {batch} algo {algo} weighted {weighted} n {n} nnz {len(ci)}", flush=True)
    kw = dict(algo=algo, iters=1, batch=batch, bht=1.0, precision=prec)
    start = x0
    for it in range(2):  # the second iteration teacher-forced from the sequential walk's first
        monkeypatch.delenv("BL_LEVELS", raising=False)
        monkeypatch.setenv("BL_WALK", "pf")
        with bl.Graph(rp, ci, w) as g:
            ref, st_ref = g.run(start, step0=0.999 ** it, **kw)
        monkeypatch.delenv("BL_WALK")
        monkeypatch.setenv("BL_LEVELS", "1")
        with bl.Graph(rp, ci, w) as g:
            got, st = g.run(start, step0=0.999 ** it, **kw)
            again, _ = g.run(start, step0=0.999 ** it, **kw)
        assert np.abs(got - ref).max() <= 1e-10 * diameter(ref), it
        assert abs(st.energy - st_ref.energy) <= 1e-10 * st_ref.energy
        assert np.array_equal(got, again)
        start = ref


@pytest.mark.parametrize("kind,batch,weighted", [("rgg", 64, False), ("rgg", 256, True), ("grid", 64, False),
                                                 ("grid", 256, True)])
def test_levels_keep_the_lagged_walks_sums(bl, monkeypatch, kind, batch, weighted):
    rp, ci = _make(kind)
    n = len(rp) - 1
    w = np.random.default_rng(7).uniform(0.5, 2.0, len(ci)).astype(np.float32) if weighted else None
    x0 = np.random.default_rng(8).random((n, 2))
    print(f"[case] levels against the lagged walk: {kind} batch {batch} weighted {weighted} n {n}", flush=True)
    out = {}
    for levels in ("0", "1"):
        monkeypatch.setenv("BL_LEVELS", levels)
        with bl.Graph(rp, ci, w) as g:
            out[levels], st = g.run(x0, algo=4, iters=3, batch=batch, bht=1.2)
            out[levels + "s"] = (st.energy, st.walk, st.walk_lag)
    assert out["0s"][1] == bl.WALK_LAG and out["1s"] == out["0s"]
    assert np.array_equal(out["0"], out["1"])
