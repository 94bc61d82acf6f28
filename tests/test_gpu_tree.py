"""The tree where its kernels' cells of 32 and 64 points, their workgroups of 256 nodes and the one-workgroup
build (2,048, 4,096 and 8,192 points) end: clusters of
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


@pytest.mark.parametrize("kind", ["clusters", "chains", "250", "254", "600", "2044", "2045", "4092", "4093", "8188", "8189"])
def test_cells_at_the_kernels_edges(bl, oracle, monkeypatch, kind):
    rng = np.random.default_rng(31)
    pts = _points(kind, rng)
    pts = pts[rng.permutation(len(pts))]
    print(f"[case] tree {kind} n {len(pts)}", flush=True)
    t, ref = bl.bh_tree(pts), oracle.bh_tree(pts)
    monkeypatch.setenv("BL_TREE_SMALL", "0")  # the general path below 8,193 points as well
    other = bl.bh_tree(pts)
    monkeypatch.delenv("BL_TREE_SMALL")
    assert all(np.array_equal(t[k], other[k]) for k in t)
    assert np.array_equal(t["perm"], ref["perm"])
    canon = [treeutil.canonical_from_child_array(x["child"], x["diam"], x["cx"], x["cy"], x.get("root", 0)) for x in (t, ref)]
    assert canon[0] == canon[1]
    for theta in (0.3, 1.2):
        assert np.array_equal(bl.bh_forces(pts, theta, precision=bl.PREC_FP64), oracle.bh_forces(pts, theta))
    if len(pts) > 5000:
        return
    want = oracle.far_forces(pts, 0.3)
    got = bl.far_forces(pts, 0.3)
    d = pts[None] - pts[:, None]
    r = np.sqrt((d * d).sum(-1))
    np.fill_diagonal(r, np.inf)
    assert np.all(np.abs(got - want).max(1) <= 1e-12 * (1.0 / r).sum(1))


@pytest.mark.parametrize("n", [700, 3000, 8000])
def test_close_pairs_in_the_one_workgroup_build(bl, oracle, n):
    """Runs of points equal in the top 48 key bits, ids not in key order."""
    rng = np.random.default_rng(n)
    base = rng.random((n // 2, 2))

    def off(k):  # at least 2^-30 per axis: distinct keys
        return rng.choice([-1.0, 1.0], (k, 2)) * rng.uniform(0.25, 1.0, (k, 2)) * 2.0**-28

    pts = np.concatenate([base, base + off(n // 2), base[:n // 8] + off(n // 8)])[:n]
    pts = pts[rng.permutation(len(pts))]
    xs, ys, _ = oracle.morton(pts)
    full = ys.astype(np.uint64) << np.uint64(32) | xs.astype(np.uint64)
    keep = np.sort(np.unique(full, return_index=True)[1])  # distinct keys
    pts = pts[keep]
    print(f"[case] close pairs n {len(pts)}", flush=True)
    t, ref = bl.bh_tree(pts), oracle.bh_tree(pts)
    assert np.array_equal(t["perm"], ref["perm"])
    assert np.array_equal(bl.bh_forces(pts, 1.2, precision=bl.PREC_FP64), oracle.bh_forces(pts, 1.2))
