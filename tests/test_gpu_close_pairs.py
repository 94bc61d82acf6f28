"""Linked pairs close together, and coincident vertices, in the all-pairs kernels of the default precision.

A linked pair has no repulsion (the reference forms its attraction only), but the dense sum adds one, which
the correction removes: the same bits, or, below 2^-40, none at all.  Three kernels: one launch a step, two
launches a step, and the batched launch (by one workgroup, and by a team).
"""
import numpy as np
import pytest

from batchlayoutcode_amd import graphs

pytestmark = pytest.mark.gpu

KERNELS = ["one", "two", "batched", "team"]


def _run(bl, monkeypatch, kernel, rp, ci, x, **kw):
    for k in ("BL_STEP_LAUNCHES", "BL_BATCHED_TEAM"):
        monkeypatch.delenv(k, raising=False)
    if kernel in ("batched", "team"):
        monkeypatch.setenv("BL_BATCHED_TEAM", "4" if kernel == "team" else "1")
        out, en, _, _ = bl.run_batched([(rp, ci)], [x], **kw)
        return out[0], en[0]
    if kernel == "two":
        monkeypatch.setenv("BL_STEP_LAUNCHES", "2")
    with bl.Graph(rp, ci) as g:
        xy, st = g.run(x, **kw)
    return xy, st.energy


def _linked(n, pairs):
    return graphs.csr_from_edges(n, np.asarray(pairs).reshape(-1, 2))


def _met(rp, ci):
    """The pairs that the reference's merge pointer meets: an empty row meets the next entry, if any."""
    n = len(rp) - 1
    m = np.zeros((n, n), bool)
    for i in range(n):
        m[i, ci[rp[i]:max(rp[i + 1], min(rp[i] + 1, rp[n]))]] = True
    return m


def _terms(x):
    """|d|^2 and the repulsion terms d/|d|^2 (0 for coincident vertices) in extended precision."""
    x = x.astype(np.longdouble)
    d = x[None, :, :] - x[:, None, :]
    r2 = (d * d).sum(-1)
    return d, r2, np.where(r2[:, :, None] > 0, d / np.where(r2 > 0, r2, 1)[:, :, None], 0)


@pytest.mark.parametrize("kernel", KERNELS)
def test_a_linked_pairs_repulsion_cancels(bl, monkeypatch, kernel):
    """One linked pair at 1e-6 .. 1e-11 without attraction, the other vertices 1e18 away: against the pair's
    term every other is below the last bit, so what the pair leaves behind is 0, or a wrong factor's
    last bits (2^-53 of 1e6 and more).  The energy is at most what the others' terms amount to."""
    rng = np.random.default_rng(1)
    print(f"[case] cancelling pair, {kernel}", flush=True)
    for n in (2, 3, 8, 9, 16, 17, 33, 250, 257, 1000, 2050):
        for d in (1e-6, 1e-8, 1e-11):
            # in the last batch: a vertex without any force left has no direction and becomes NaN
            a, b = (n - 1) // 1024 * 1024 + rng.choice((n - 1) % 1024 + 1, 2, replace=False)
            phi = rng.random(n) * 2 * np.pi
            x = 1e18 * (1 + rng.random(n))[:, None] * np.stack([np.cos(phi), np.sin(phi)], 1)
            x[a] = rng.random(2)
            x[b] = x[a] + d * np.array([np.cos(phi[0]), np.sin(phi[0])])
            rp, ci = _linked(n, [(a, b)])
            xy, e = _run(bl, monkeypatch, kernel, rp, ci, x, algo=8, iters=1, weight=0.0, batch=1024, step0=1e-200)
            _, _, t = _terms(x)
            t[_met(rp, ci)] = 0
            most = np.sqrt((t * t).sum(-1)).sum(1)
            assert e <= 2 * float((most * most).sum()), (n, d, e)
            if n == 2:  # no force: no direction either, as in the reference
                assert e == 0.0 and np.isnan(xy).all()


@pytest.mark.parametrize("law", [2, 8])
@pytest.mark.parametrize("kernel", KERNELS)
def test_force_of_linked_pairs_closer_than_rounding(bl, monkeypatch, kernel, law):
    """Linked pairs at 1e-13 .. 1e-20 around the origin among vertices in the unit box (one of them linked to
    more vertices than one correction piece takes): |F| in extended precision, to (n + 16) roundings of the
    terms that the reference forms."""
    eps = 2.0 ** -53
    rng = np.random.default_rng(2)
    for n, d in ((2, 1e-15), (9, 1e-13), (40, 1e-16), (300, 1e-18), (1000, 1e-15), (1024, 1e-20)):
        print(f"[case] close pair, {kernel} law {law} n {n} distance {d}", flush=True)
        x = 0.05 + rng.random((n, 2))
        a, b = rng.choice(n, 2, replace=False)
        phi = rng.random() * 2 * np.pi
        x[a] = 0.0
        x[b] = d * np.array([np.cos(phi), np.sin(phi)])
        pairs = [(a, b)] + [(a, k) for k in range(n) if k not in (a, b) and (n == 1000 or k % 5 == 0)]
        rp, ci = _linked(n, pairs)
        kw = dict(algo=law, iters=1, weight=0.7, batch=1024, step0=1.0)
        xy, e = _run(bl, monkeypatch, kernel, rp, ci, x, **kw)
        diff, r2, t = _terms(x)
        met = _met(rp, ci)
        t[met] = 0
        att = np.where(met, np.longdouble(0.7) * (np.sqrt(r2) if law == 2 else 1), 0)
        terms = att[:, :, None] * diff - t
        F = terms.sum(1)
        mag = np.sqrt((F * F).sum(-1))
        # a linked vertex further away than 2^-40 is still added and removed
        both = np.where(r2 > 0, 1 / np.sqrt(np.where(r2 > 0, r2, 1)), 0) * met * (r2 >= 2.0 ** -80)
        tot = np.sqrt((terms * terms).sum(-1)).sum(1) + 2 * both.sum(1)
        if n == 2:
            assert np.abs(e - (mag * mag).sum()) <= 1e-14 * (mag * mag).sum()
        err = (n + 16) * eps * tot / mag
        got = xy.astype(np.longdouble) - x
        bound = 2 * err + 8 * eps * (1 + np.abs(x).max(1))
        worst = (np.abs(got - F / mag[:, None]).max(1) / bound).max()
        assert worst <= 1.0, (n, d, float(worst))


@pytest.mark.parametrize("kernel", KERNELS)
def test_coincident_vertices_in_one_group(bl, monkeypatch, kernel):
    """5, 6, 8 and 20 vertices in the same place with consecutive ids: the product of a group's |d|^2
    underflows, and its pairs have factors of their own.  Coincident pairs add nothing."""
    eps = 2.0 ** -53
    rng = np.random.default_rng(3)
    for n, m in ((24, 5), (24, 6), (40, 8), (300, 20), (1000, 6)):
        print(f"[case] coincident, {kernel} n {n} of them {m}", flush=True)
        x = rng.random((n, 2))
        x[8:8 + m] = x[8]
        rp, ci = _linked(n, [(8, 9), (9, n - 1)])
        xy, e = _run(bl, monkeypatch, kernel, rp, ci, x, algo=8, iters=1, weight=1.0, batch=1024, step0=1.0)
        diff, r2, t = _terms(x)
        met = _met(rp, ci)
        both = np.sqrt((t * t).sum(-1)) * met
        t[met] = 0
        terms = met[:, :, None] * diff - t
        F = terms.sum(1)
        mag = np.sqrt((F * F).sum(-1))
        tot = np.sqrt((terms * terms).sum(-1)).sum(1) + 2 * both.sum(1)
        got = xy.astype(np.longdouble) - x
        bound = 2 * (n + 16) * eps * tot / mag + 8 * eps * (1 + np.abs(x).max(1))
        worst = (np.abs(got - F / mag[:, None]).max(1) / bound).max()
        assert worst <= 1.0, (n, m, float(worst))


@pytest.mark.parametrize("kernel", KERNELS)
def test_all_vertices_in_a_tiny_ball(bl, monkeypatch, kernel):
    """Every pair is closer than 2^-40, linked or not: a vertex's neighbours, up to all others, are found among
    them all.  No attraction: |F| against extended precision as above."""
    eps = 2.0 ** -53
    rng = np.random.default_rng(4)
    for n, deg in ((7, 2), (130, 4), (1000, 9), (1024, 40)):
        print(f"[case] tiny ball, {kernel} n {n} degree {deg}", flush=True)
        x = 1e-14 * rng.random((n, 2))
        e = np.concatenate([rng.integers(0, n, (n * deg // 2, 2)), np.stack([np.full(n, n // 2), np.arange(n)], 1)])
        e = np.unique(np.sort(e[e[:, 0] != e[:, 1]], 1), axis=0)
        e = e[~((e == 0).any(1) & (e == n // 2).any(1))]  # the hub keeps one repulsion: a direction
        rp, ci = _linked(n, e)
        xy, en = _run(bl, monkeypatch, kernel, rp, ci, x, algo=8, iters=1, weight=0.0, batch=1024, step0=1e-14)
        _, _, t = _terms(x)
        t[_met(rp, ci)] = 0
        F = -t.sum(1)
        mag = np.sqrt((F * F).sum(-1))
        tot = np.sqrt((t * t).sum(-1)).sum(1)
        got = (xy.astype(np.longdouble) - x) / 1e-14
        bound = 2 * (n + 16) * eps * tot / mag + 16 * eps
        worst = (np.abs(got - F / mag[:, None]).max(1) / bound).max()
        assert worst <= 1.0, (n, float(worst))
