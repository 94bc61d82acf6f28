"""The tree where its kernels' cells of 32 and 64 points and their workgroups of 256 nodes end: clusters of
31..65 points, chains as deep as a small cell can be, points at the frame's last key.  Tree and FP64
forces bit for bit the oracle's; the far field's (whose cells are summed by other routes) to 1e-12 of
the terms' magnitudes."""
import numpy as np
import pytest

import treeutil

pytestmark = pytest.mark.gpu


def _points(kind, rng):
    if kind == "clusters":
        sizes = [31, 32, 33, 34, 63, 64, 65] * 8
        p = [c + 1e-4 * rng.random((m, 2)) for c, m in zip(rng.random((len(sizes), 2)), sizes)]
        return np.concatenate(p)
    if kind == "chains":  # a chain halves its cell towards a corner point by point
        t = 0.5 ** np.arange(1, 26)[:, None]
        p = [c + 2.0**-4 * t * (0.9 + 0.1 * rng.random((25, 2))) * s
             for c, s in zip(rng.random((40, 2)), rng.choice([-1.0, 1.0], (40, 1, 2)))]
        return np.concatenate(p)
    return np.concatenate([rng.random((int(kind), 2)), [[1.0, 1.0], [1.0, 0.0], [0.0, 0.0], [0.0, 1.0]]])


@pytest.mark.parametrize("kind", ["clusters", "chains", "250", "254", "600"])
def test_cells_at_the_kernels_edges(bl, oracle, kind):
    rng = np.random.default_rng(31)
    pts = _points(kind, rng)
    pts = pts[rng.permutation(len(pts))]
    print(f"[case] tree {kind} n {len(pts)}", flush=True)
    t, ref = bl.bh_tree(pts), oracle.bh_tree(pts)
    assert np.array_equal(t["perm"], ref["perm"])
    canon = [treeutil.canonical_from_child_array(x["child"], x["diam"], x["cx"], x["cy"], x.get("root", 0)) for x in (t, ref)]
    assert canon[0] == canon[1]
    for theta in (0.3, 1.2):
        assert np.array_equal(bl.bh_forces(pts, theta, precision=bl.PREC_FP64), oracle.bh_forces(pts, theta))
    want = oracle.far_forces(pts, 0.3)
    got = bl.far_forces(pts, 0.3)
    d = pts[None] - pts[:, None]
    r = np.sqrt((d * d).sum(-1))
    np.fill_diagonal(r, np.inf)
    assert np.all(np.abs(got - want).max(1) <= 1e-12 * (1.0 / r).sum(1))
