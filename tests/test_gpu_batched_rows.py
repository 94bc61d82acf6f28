"""Batched launch: the neighbours met in unsorted rows (a row's strictly increasing prefix; an empty row
takes the next row's first entry, none at the end of the graph) at the widths its kernel loads them in,
against the oracle on each graph alone to the bound of the batched launch's oracle tests."""
import numpy as np
import pytest

from conftest import diameter

pytestmark = pytest.mark.gpu


def _graph(rng, n, kind):
    rows = []
    for i in range(n):
        m = {"short": i % 20, "hub": n if i == 3 else i % 3, "empty": 0 if i % 4 or i > n - 4 else 9}[kind]
        row = np.sort(rng.choice(n, min(m, n), replace=False))
        if kind != "hub" and len(row) > 1:
            k = i % len(row)  # a descent, or a repeated entry, before place k
            row = np.concatenate([row[:k], row[k:][::-1] if i % 2 else np.repeat(row[k:], 2)])
        rows.append(row)
    rp = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int32)
    return rp, np.concatenate(rows).astype(np.int32)


@pytest.mark.parametrize("n", [33, 300, 2100])
def test_rows_as_the_reference_meets_them(bl, oracle, n):
    rng = np.random.default_rng(n)
    gs = [_graph(rng, n, kind) for kind in ("short", "hub", "empty")]
    xys = [rng.random((n, 2)) for _ in gs]
    print(f"[case] batched rows n {n}", flush=True)
    out, en, _, _ = bl.run_batched(gs, xys, algo=2, iters=1, batch=64)
    for (rp, ci), x0, xy, e in zip(gs, xys, out, en):
        ref, e_ref, _ = oracle.minibatch(rp, ci, x0, 1, 64)
        assert np.abs(xy - ref).max() <= 1e-8 * diameter(ref)
        assert abs(e - e_ref) <= 1e-8 * e_ref
