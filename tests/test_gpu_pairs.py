"""The dense repulsion's groups of eight pairs at the sizes where groups, loads and chunks end.

One Jacobi step with no attraction (algo 8, weight 0, one batch): x' - x = F/|F| and energy =
sum |F|^2, F the repulsion.  Against numpy in extended precision the force's error is at most
(n + 16) roundings of 2^-53 of sum_j |term_j| (n additions; the difference, |d|^2, eight products, the
reciprocal and the product take fewer than 16), so the unit vector's is that over |F|, twice
(numerator and norm), plus a few roundings of the position itself.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [2, 3, 7, 8, 9, 15, 16, 17, 31, 33, 63, 65, 127, 130, 257, 1000, 1024]


def _forces(x):
    x = x.astype(np.longdouble)
    d = x[None, :, :] - x[:, None, :]
    r2 = (d * d).sum(-1)
    np.fill_diagonal(r2, 1)
    t = d / r2[:, :, None]
    return -t.sum(1), np.sqrt((t * t).sum(-1)).sum(1)


@pytest.mark.parametrize("scale", [1.0, 1e-7, 1e12, 1e40])
@pytest.mark.parametrize("batched", [False, True])
def test_groups_of_pairs(bl, scale, batched):
    """1e40: a group's product of |d|^2 leaves the FP64 range, the pairs are taken one by one."""
    eps = 2.0 ** -53
    graphs, xs = [], []
    for n in SIZES:
        graphs.append((np.zeros(n + 1, np.int32), np.zeros(0, np.int32)))
        xs.append(np.random.default_rng(n).random((n, 2)) * scale)
    kw = dict(algo=8, iters=1, weight=0.0, batch=1024, step0=scale)
    if batched:
        out, en, _, _ = bl.run_batched(graphs, xs, **kw)
    else:
        out, en = [], []
        for k in range(len(SIZES)):
            with bl.Graph(*graphs[k]) as g:
                xy, st = g.run(xs[k], **kw)
            out.append(xy)
            en.append(st.energy)
    for k, xy, e in zip(range(len(SIZES)), out, en):
        n = SIZES[k]
        F, tot = _forces(xs[k])
        mag = np.sqrt((F * F).sum(1))
        err = (n + 16) * eps * tot / mag  # relative error of F
        got = (xy.astype(np.longdouble) - xs[k]) / scale
        bound = 2 * err + 8 * eps * (1 + np.abs(xs[k]).max(1) / scale)
        worst = np.abs(got - F / mag[:, None]).max(1) / bound
        assert worst.max() <= 1.0, (n, float(worst.max()))
        E = (mag * mag).sum()
        assert abs(e - E) <= 2 * (err * mag * mag).sum() + (n + 8) * eps * E, n
