"""The training kernels where their 16-sample tiles and 64-sample workgroups end: loss and gradient against
the CPU reference with BF16 products (the bounds of the model's other gradient test), and a batch's Adam
step against the same step on the host from that gradient."""
import numpy as np
import pytest

from oracle import mlp_ref as M

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 129, 1040])
def test_gradient_and_step_at_the_tiles_ends(bl, n):
    rng = np.random.default_rng(n)
    p = bl.far_model_init(3)
    p[M.OFFSETS["W4"][0]:M.OFFSETS["W4"][0] + 128] *= 10
    X = rng.standard_normal((n, 8)).astype(np.float32)
    T = (0.1 * rng.standard_normal((n, 2))).astype(np.float32)
    print(f"[case] mlp tiles n {n}", flush=True)
    loss, g = bl.far_model_grad(p, X, T)
    rl, rg = M.loss_grad(p, X, T, emulate=True)
    assert abs(loss - rl) <= 1e-3 * rl
    for k, (o, s) in M.OFFSETS.items():
        m = int(np.prod(s))
        assert np.linalg.norm(g[o:o + m] - rg[o:o + m]) <= 1e-2 * np.linalg.norm(rg[o:o + m]), k
    p1, losses = bl.far_model_train(p, X, T, epochs=1, batch=n, lr=1e-3, seed=1)
    assert abs(losses[0] - loss) <= 1e-5 * loss
    # the first step of Adam moves a parameter by lr g / (|g| + eps), whatever the samples' order did to g
    big = np.abs(g) > 1e-3 * np.abs(g).max()
    assert np.abs((p1 - p)[big] + 1e-3 * np.sign(g[big])).max() <= 1e-5
