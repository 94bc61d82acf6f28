"""The tree traversals where their stack and their sums can go wrong: trees so deep that the pending
siblings exceed the stack's registers, waves with few queries, single and coincident queries.

A traversal that lost or repeated an entry would be off by whole terms.  Bars: unit vectors carry at
most 2^-48 relative error each and their sum of at most n terms n roundings, n (2^-48 + n 2^-53); the
monopoles 1e-12 of sum_j 1/|x_j - q| (the far field's bar).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _nested(levels, rng):
    """Points in the three outer quadrants of cells nested towards the origin: every level leaves
    three siblings waiting while the first quadrant is descended."""
    s = 2.0 ** -np.arange(levels)[:, None, None]
    at = np.array([[1.5, 0.5], [0.5, 1.5], [1.5, 1.5]])[None] + 0.2 * rng.random((levels, 3, 2))
    return np.concatenate([(0.5 * s * at).reshape(-1, 2), [[0.0, 0.0], [1.0, 1.0]]])


def _case(kind):
    rng = np.random.default_rng(3)
    if kind == "nested":
        return _nested(29, rng)
    if kind == "nested_dense":
        return np.concatenate([_nested(27, rng), rng.random((500, 2)), 2.0 ** -20 * rng.random((200, 2))])
    if kind == "two":
        return rng.random((2, 2))
    return rng.random((65, 2))


@pytest.mark.parametrize("kind", ["nested", "nested_dense", "two", "65"])
@pytest.mark.parametrize("theta", [0.0, 0.37, 1.13])
def test_deep_trees(bl, oracle, kind, theta):
    xy = _case(kind)
    q = np.concatenate([xy, np.random.default_rng(4).random((3, 2))])
    n = len(xy)
    print(f"[case] traversal {kind} theta {theta} n {n}", flush=True)
    got = bl.bh_forces(xy, theta, q, precision=bl.PREC_MIXED)
    ref = oracle.bh_forces(xy, theta, q)
    assert np.abs(got - ref).max() <= n * (2.0 ** -48 + n * 2.0 ** -53)
    d = np.sqrt(((xy[None] - q[:, None]) ** 2).sum(-1))
    scale = np.where(d > 0, 1.0 / np.where(d > 0, d, 1.0), 0.0).sum(1)
    got = bl.far_forces(xy, theta, queries=q)
    ref = oracle.far_forces(xy, theta, q)
    assert np.all(np.abs(got - ref).max(1) <= 1e-12 * scale)
