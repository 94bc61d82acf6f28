"""The level walk's plan takes device memory only where the levels are chosen, and a plan that there is no
memory for leaves none behind: the walk in its place runs, with the same layout."""
import numpy as np
import pytest
import torch

from batchlayoutcode_amd import graphs

pytestmark = pytest.mark.gpu


def _taken(g, x0, **kw):
    """Device memory that a run took beyond what was there before it."""
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    out = g.run(x0, algo=4, iters=1, bht=1.2, **kw)
    torch.cuda.synchronize()
    return before - torch.cuda.mem_get_info()[0], out


def test_rejected_levels_take_no_memory(bl, monkeypatch):
    """A grid in row order at -batch 256: the lagged walk is the faster one."""
    rp, ci = graphs.csr_from_edges(*graphs.grid(700, 700))
    x0 = np.random.default_rng(8).random((len(rp) - 1, 2))
    print("[case] plan of levels that are not chosen", flush=True)
    monkeypatch.delenv("BL_LEVELS", raising=False)
    with bl.Graph(rp, ci) as g:  # the library's first use
        g.run(x0, algo=4, iters=1, batch=256)
    taken = {}
    for levels in ("0", None):
        if levels:
            monkeypatch.setenv("BL_LEVELS", levels)
        else:
            monkeypatch.delenv("BL_LEVELS")
        with bl.Graph(rp, ci) as g:
            taken[levels], (_, st) = _taken(g, x0, batch=256)
            assert st.walk == bl.WALK_LAG and st.walk_levels == 0
    assert taken[None] == taken["0"], taken


@pytest.mark.parametrize("kind,batch,walk", [("rgg", 64, "LAG"), ("rmat", 1024, "WIDE")])
def test_no_memory_for_the_plan(bl, monkeypatch, kind, batch, walk):
    rp, ci = (graphs.csr_from_edges(*graphs.rgg(120_000, seed=5)) if kind == "rgg" else
              graphs.csr_from_edges(*graphs.rmat(15, 8, seed=2)[:2]))
    x0 = np.random.default_rng(8).random((len(rp) - 1, 2))
    print(f"[case] no memory for the plan, {kind}", flush=True)
    monkeypatch.setenv("BL_LEVELS", "0")
    with bl.Graph(rp, ci) as g:  # the kernels' first use
        g.run(x0, algo=4, iters=1, batch=batch)
    with bl.Graph(rp, ci) as g:
        taken, (ref, st) = _taken(g, x0, batch=batch)
        assert st.walk == getattr(bl, "WALK_" + walk)
    monkeypatch.delenv("BL_LEVELS")
    monkeypatch.setenv("BL_LEVEL_PAD_GIB", "4096")
    with bl.Graph(rp, ci) as g:
        same, (xy, st) = _taken(g, x0, batch=batch)
        assert st.walk == getattr(bl, "WALK_" + walk) and st.walk_levels == 0
        assert np.array_equal(xy, ref) and same == taken
        monkeypatch.delenv("BL_LEVEL_PAD_GIB")
        assert np.array_equal(g.run(x0, algo=4, iters=1, bht=1.2, batch=batch)[0], ref)  # the refusal is kept
