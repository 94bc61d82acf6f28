"""The level walk keeps the arithmetic of the walk that it stands for.

Where the row walk is chosen for a graph, the levels form the same sums with the same roots and divisions, so
rows of up to 16 early entries (and their late sums) come out bit for bit; where the lagged walk is chosen,
all rows do, also those with more late entries than the other graphs' slices hold (32).
"""
import numpy as np
import pytest

from batchlayoutcode_amd import graphs

pytestmark = pytest.mark.gpu


def _path_in_any_order(n, seed):
    p = np.random.default_rng(seed).permutation(n)
    return np.stack([p[:-1], p[1:]], 1)


def _make(kind):
    if kind.startswith("path"):
        n = int(kind[4:])
        return graphs.csr_from_edges(n, _path_in_any_order(n, 1))
    if kind.startswith("grid"):  # natural order: levels for k_level_run
        return graphs.csr_from_edges(*graphs.grid(int(kind[4:]), int(kind[4:])))
    n, e = graphs.rgg(2200, seed=5)  # no more than 16 edges from a vertex to smaller ids
    e = e[np.argsort(e.max(1), kind="stable")]
    hi = e.max(1)
    at = np.arange(len(e))
    first = np.concatenate([[True], hi[1:] != hi[:-1]])
    return graphs.csr_from_edges(n, e[at - np.maximum.accumulate(np.where(first, at, 0)) < 16])


@pytest.mark.parametrize("kind,batch,weighted", [("path2000", 256, False), ("path130", 16, True), ("grid45", 256, True),
                                                 ("grid30", 100, False), ("grid30", 100, True), ("rgg", 256, True),
                                                 ("rgg", 256, False)])
def test_row_walks_bits(bl, monkeypatch, kind, batch, weighted):
    rp, ci = _make(kind)
    n = len(rp) - 1
    w = np.random.default_rng(7).uniform(0.5, 2.0, len(ci)).astype(np.float32) if weighted else None
    x0 = np.random.default_rng(8).random((n, 2))
    print(f"[case] levels against the row walk: {kind} batch {batch} weighted {weighted} n {n} nnz {len(ci)}", flush=True)
    out = {}
    for levels in ("0", "1"):
        monkeypatch.setenv("BL_LEVELS", levels)
        with bl.Graph(rp, ci, w) as g:
            out[levels], st = g.run(x0, algo=4, iters=3, batch=batch, bht=1.0)
            assert st.walk == bl.WALK_ROW, (levels, st.walk)
    assert np.array_equal(out["0"], out["1"])


@pytest.mark.parametrize("weighted", [False, True])
def test_lagged_walks_bits_with_long_late_rows(bl, monkeypatch, weighted):
    """40 vertices of the first batch with 33 to 62 neighbours each, all of them in later batches."""
    n = 20_000
    rng = np.random.default_rng(3)
    e = [_path_in_any_order(n, 1)]
    for k in range(40):
        others = rng.choice(np.arange(64, n), 33 + k * 28 // 40, replace=False)
        e.append(np.stack([np.full(len(others), k), others], 1))
    e = np.unique(np.sort(np.concatenate(e), 1), axis=0)
    rp, ci = graphs.csr_from_edges(n, e)
    w = np.random.default_rng(7).uniform(0.5, 2.0, len(ci)).astype(np.float32) if weighted else None
    x0 = np.random.default_rng(8).random((n, 2))
    print(f"[case] levels against the lagged walk, long late rows, weighted {weighted}", flush=True)
    out = {}
    for levels in ("0", "1"):
        monkeypatch.setenv("BL_LEVELS", levels)
        with bl.Graph(rp, ci, w) as g:
            out[levels], st = g.run(x0, algo=4, iters=3, batch=64, bht=1.0)
            assert st.walk == bl.WALK_LAG
    assert np.array_equal(out["0"], out["1"])
