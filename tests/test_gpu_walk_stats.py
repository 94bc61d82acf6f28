"""Which batch walk ran: bl_stats.walk_levels, and the walks that the levels replace by default, run themselves
(BL_LEVELS=0) against the oracle and against each other."""
import numpy as np
import pytest

from batchlayoutcode_amd import graphs
from conftest import diameter

pytestmark = pytest.mark.gpu


def _levels(rp, ci, B):
    """The dependence levels of the batches: one more than the highest level of a neighbour in an earlier one."""
    n = len(rp) - 1
    lev = np.zeros(n, np.int64)
    rows = np.repeat(np.arange(n), np.diff(rp))
    for b0 in range(0, n, B):
        s, e = rp[b0], rp[min(n, b0 + B)]
        early = ci[s:e] < b0
        np.maximum.at(lev, rows[s:e][early], lev[ci[s:e][early]] + 1)
    return int(lev.max()) + 1


def _make(kind):
    if kind == "rgg":
        return graphs.csr_from_edges(*graphs.rgg(30_000, seed=5))
    if kind == "grid":
        return graphs.csr_from_edges(*graphs.grid(70, 300))
    if kind == "path":
        i = np.arange(2999)
        return graphs.csr_from_edges(3000, np.stack([i, i + 1], 1))
    return graphs.csr_from_edges(*graphs.rmat(13, 8, seed=2)[:2])


@pytest.mark.parametrize("kind,batch", [("rgg", 64), ("rgg", 256), ("grid", 64), ("path", 64), ("rmat", 100), ("rmat", 1024),
                                        ("rmat", 3000)])
def test_levels_are_reported(bl, monkeypatch, kind, batch):
    rp, ci = _make(kind)
    x0 = np.random.default_rng(8).random((len(rp) - 1, 2))
    print(f"[case] levels reported: {kind} batch {batch}", flush=True)
    kw = dict(iters=1, batch=batch, bht=1.2)
    with bl.Graph(rp, ci) as g:
        monkeypatch.setenv("BL_LEVELS", "1")
        assert g.run(x0, algo=4, **kw)[1].walk_levels == _levels(rp, ci, batch)
        assert g.run(x0, algo=4, precision=bl.PREC_FP64, **kw)[1].walk_levels == 0
        assert g.run(x0, algo=2, **kw)[1].walk_levels == 0
        monkeypatch.setenv("BL_LEVELS", "0")
        st = g.run(x0, algo=4, **kw)[1]
        assert st.walk_levels == 0 and st.walk != bl.WALK_NONE
        monkeypatch.delenv("BL_LEVELS")
        assert g.run(x0, algo=4, **kw)[1].walk_levels in (0, _levels(rp, ci, batch))


@pytest.mark.parametrize("batch", [64, 256])
def test_lagged_walk_and_its_helpers(bl, monkeypatch, batch):
    rp, ci = graphs.csr_from_edges(*graphs.delaunay_holes(100_000, seed=3))
    x0 = np.random.default_rng(8).random((len(rp) - 1, 2))
    print(f"[case] lagged walk itself, batch {batch}", flush=True)
    monkeypatch.setenv("BL_LEVELS", "0")
    out = {}
    for mode, env in (("lag", {}), ("alone", dict(BL_LAG_H="0")), ("row", dict(BL_WALK="row"))):
        for k in ("BL_LAG_H", "BL_WALK"):
            monkeypatch.delenv(k, raising=False)
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        with bl.Graph(rp, ci) as g:
            out[mode] = g.run(x0, algo=4, iters=1, batch=batch, bht=1.2)
        assert out[mode][1].walk_levels == 0
    assert out["lag"][1].walk == bl.WALK_LAG and out["lag"][1].walk_helped > 0 and out["alone"][1].walk_helped == 0
    assert np.array_equal(out["lag"][0], out["alone"][0])
    assert np.abs(out["lag"][0] - out["row"][0]).max() <= 1e-10 * diameter(out["row"][0])


@pytest.mark.parametrize("levels", ["0", None])
def test_rmat_wide_walk_and_levels_vs_oracle(bl, oracle, monkeypatch, levels):
    """The wide walk itself and the levels in its place: iteration 1 and a teacher-forced iteration 2 within
    1e-4 of the oracle's diameter and energy."""
    n, e, w = graphs.rmat(15, 8, seed=2)
    rp, ci, w = graphs.csr_from_edges(n, e, w)
    x0 = graphs.uniform_init(n, 0)
    monkeypatch.delenv("BL_WALK", raising=False)
    monkeypatch.delenv("BL_LEVELS", raising=False)
    if levels:
        monkeypatch.setenv("BL_LEVELS", levels)
    print(f"[case] rmat15 algo 4 batch 1024 BL_LEVELS {levels}", flush=True)
    start = x0
    with bl.Graph(rp, ci, w) as g:
        for it in range(2):
            ref, e_ref = oracle.bh_layout(rp, ci, start, 1, 1024, theta=1.2, step0=0.999 ** it, w_edge=w)
            x, st = g.run(start, algo=4, iters=1, batch=1024, bht=1.2, step0=0.999 ** it)
            assert st.walk == bl.WALK_WIDE and (st.walk_levels == 0) == (levels == "0")
            assert np.abs(x - ref).max() <= 1e-4 * diameter(ref)
            assert abs(st.energy - e_ref) <= 1e-4 * e_ref
            start = ref
