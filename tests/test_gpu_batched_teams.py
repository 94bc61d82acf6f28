"""Batched launch: a graph laid out by a team of workgroups gets the same bits as by one."""
import numpy as np
import pytest

from batchlayoutcode_amd import graphs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def bl():
    from batchlayoutcode_amd import api

    return api


# a graph of one vertex (its zero force has no direction: NaN, as in the oracle), sizes at the edges of the chunk counts (2,048 and 4,096), a last batch of one vertex, graphs smaller than
# a batch, and the largest size
SIZES = [1, 63, 129, 2047, 2048, 2049, 4095, 4097, 8192, 300]


@pytest.mark.parametrize("batch", [1, 64, 128, 1000])
def test_teams_give_the_same_bits(bl, monkeypatch, batch):
    rng = np.random.default_rng(batch)
    sizes = SIZES if batch > 1 else [1, 63, 129, 300]
    gs = []
    for n in sizes:
        e = rng.integers(0, n, (4 * n, 2))
        gs.append(graphs.csr_from_edges(n, e[e[:, 0] != e[:, 1]]))
    xys = [rng.random((n, 2)) for n in sizes]
    kw = dict(algo=2, iters=3, batch=batch)
    monkeypatch.setenv("BL_BATCHED_TEAM", "1")
    ref, en, _, _ = bl.run_batched(gs, xys, **kw)
    # 0: a first wait that ends at once, after which a launch without teams takes the graphs over
    for team, wait in (("2", None), ("4", None), ("8", None), ("16", None), ("8", "0"), (None, None)):
        for k, v in (("BL_BATCHED_TEAM", team), ("BL_BATCHED_WAIT_US", wait)):
            monkeypatch.delenv(k, raising=False) if v is None else monkeypatch.setenv(k, v)
        print(f"[case] team {team} wait {wait}", flush=True)
        out, en_t, fin, _ = bl.run_batched(gs, xys, **kw)
        assert all(np.array_equal(a, b, equal_nan=True) for a, b in zip(out, ref)), (team, wait)
        assert np.array_equal(en, en_t, equal_nan=True) and (fin > 0).all(), (team, wait)
