"""The sort whose workgroups sum the tiles' counts themselves, where its tiles (2,048 keys), its waves' shares of
them (4 and 64 tiles) and its range (128 tiles) end: the same order as with the scan's launch, and the
oracle's where that is quick."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [8193, 10240, 10241, 18432, 131072, 131073, 262143, 262144, 262145])
def test_same_order_with_and_without_the_scan(bl, oracle, monkeypatch, n):
    rng = np.random.default_rng(n)
    pts = rng.random((n, 2))
    pts[: n // 3] = 0.3 + 1e-3 * pts[: n // 3]  # most of a pass's keys in a few digits
    print(f"[case] sort n {n}", flush=True)
    t = bl.bh_tree(pts)
    monkeypatch.setenv("BL_SORT_SUM", "0")
    other = bl.bh_tree(pts)
    assert all(np.array_equal(t[k], other[k]) for k in t)
    if n < 20000:
        assert np.array_equal(t["perm"], oracle.bh_tree(pts)["perm"])
