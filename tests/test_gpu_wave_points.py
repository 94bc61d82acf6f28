"""A traversal's forces don't depend on how many points share a wave."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 7, 63, 65, 1000, 5001])
def test_forces_are_the_same_bits(bl, monkeypatch, n):
    rng = np.random.default_rng(n)
    pts = rng.random((n, 2))
    pts[n // 2:] = 0.3 + 0.01 * pts[n // 2:]
    q = np.concatenate([pts[::3], rng.random((17, 2))])
    runs = {}
    for per in ("64", "32", "16", "8", None):
        monkeypatch.delenv("BL_WAVE_POINTS", raising=False)
        if per:
            monkeypatch.setenv("BL_WAVE_POINTS", per)
        print(f"[case] wave points n {n} per {per}", flush=True)
        runs[per] = [bl.bh_forces(pts, 0.9, precision=bl.PREC_MIXED), bl.bh_forces(pts, 0.9, precision=bl.PREC_FP32),
                     bl.bh_forces(pts, 1.2, queries=q, precision=bl.PREC_MIXED), bl.far_forces(pts, 0.4),
                     bl.far_forces(pts, 0.8, mode=bl.FAR_QUAD, queries=q)]
    for per, out in runs.items():
        assert all(np.array_equal(a, b) for a, b in zip(out, runs["64"])), per
