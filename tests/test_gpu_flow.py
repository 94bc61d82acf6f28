"""The level walk's launches of several levels (ordered by the positions themselves) and its one-workgroup
runs, in turn within one iteration: against the sequential walk to 1e-10 of the diameter, the bar of the
other walks.  And its waits: past their deadline a run ends with an error, and the next one is whole.
"""
import numpy as np
import pytest

from batchlayoutcode_amd import graphs
from conftest import diameter

pytestmark = pytest.mark.gpu


def _chain_and_crowd(crowd, hub):
    """A path 0 .. 599 (runs of levels of one or two vertices); `crowd` vertices on its vertex 300 (one level
    for k_level_flow); one vertex on `hub` of them (a row of that length in the next level); a path from
    that one (a run that starts from a level of k_level_flow)."""
    n0 = 600
    i = np.arange(n0 - 1)
    c = n0 + np.arange(crowd)
    h = n0 + crowd
    t = np.arange(h, h + 40)
    e = [np.stack([i, i + 1], 1), np.stack([np.full(crowd, 300), c], 1), np.stack([c[:hub], np.full(hub, h)], 1),
         np.stack([t, t + 1], 1)]
    return graphs.csr_from_edges(h + 41, np.concatenate(e))


@pytest.mark.parametrize("crowd,hub,batch,weighted", [
    (2049, 9, 1, False), (2200, 64, 3, True), (4096, 512, 1, True), (3000, 513, 2, False), (6000, 5000, 7, True)])
def test_launches_and_runs_in_turn(bl, monkeypatch, crowd, hub, batch, weighted):
    rp, ci = _chain_and_crowd(crowd, hub)
    n = len(rp) - 1
    w = np.random.default_rng(7).uniform(0.5, 2.0, len(ci)).astype(np.float32) if weighted else None
    x0 = np.random.default_rng(8).random((n, 2))
    print(f"[case] flow crowd {crowd} hub {hub} batch {batch} weighted {weighted} n {n}", flush=True)
    kw = dict(algo=4, iters=1, batch=batch, bht=1.0)
    monkeypatch.setenv("BL_WALK", "pf")
    with bl.Graph(rp, ci, w) as g:
        ref, st_ref = g.run(x0, **kw)
    monkeypatch.delenv("BL_WALK")
    monkeypatch.setenv("BL_LEVELS", "1")
    with bl.Graph(rp, ci, w) as g:
        got, st = g.run(x0, **kw)
        again, _ = g.run(x0, **dict(kw, iters=3))
        twice, _ = g.run(x0, **dict(kw, iters=3))
    assert np.abs(got - ref).max() <= 1e-10 * diameter(ref)
    assert abs(st.energy - st_ref.energy) <= 1e-10 * st_ref.energy
    assert np.array_equal(again, twice)


def test_a_wait_past_its_deadline_is_an_error(bl, monkeypatch):
    rp, ci = graphs.csr_from_edges(*graphs.rmat(13, 8, seed=2)[:2])
    x0 = np.random.default_rng(8).random((len(rp) - 1, 2))
    kw = dict(algo=4, iters=2, batch=100, bht=1.0)
    print(f"[case] flow deadline n {len(rp) - 1}", flush=True)
    monkeypatch.setenv("BL_LEVELS", "1")
    with bl.Graph(rp, ci) as g:
        ref, _ = g.run(x0, **kw)
        monkeypatch.setenv("BL_LEVEL_WAIT_US", "-1")  # gives up at the first wait
        with pytest.raises(bl.BLError):
            g.run(x0, **kw)
        monkeypatch.delenv("BL_LEVEL_WAIT_US")
        got, _ = g.run(x0, **kw)
    assert np.array_equal(got, ref)
