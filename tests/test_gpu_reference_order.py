"""FP64 mode at the edges of its blocks: 512 positions a block, 64 a tile, 16 vertices a row, more than 64
neighbours of a vertex in one block and over several, coincident points.  The strict-IEEE oracle's
coordinates and energy bit for bit (LinLog, whose logarithm is the device's, to 1e-10 of the diameter)."""
import numpy as np
import pytest

from batchlayoutcode_amd import graphs
from conftest import diameter

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch", [(511, 15), (512, 16), (513, 17), (1025, 200), (1601, 256), (2500, 1000)])
def test_blocks_tiles_and_hubs(bl, oracle, n, batch):
    rng = np.random.default_rng(n)
    e = [rng.integers(0, n, (4 * n, 2)), np.stack([np.full(n, 7), np.arange(n)], 1)]  # 7: a neighbour of all
    e += [np.stack([np.full(300, n - 1), rng.choice(n, 300, replace=False)], 1)]
    e = np.concatenate(e)
    rp, ci = graphs.csr_from_edges(n, e[e[:, 0] != e[:, 1]])
    w = rng.uniform(0.5, 2.0, len(ci)).astype(np.float32)
    init = rng.random((n, 2))
    init[n // 2] = init[3]
    for law in (2, 3, 8):
        for we in (None, w):
            print(f"[case] n {n} batch {batch} law {law} weights {we is not None}", flush=True)
            ref, e_ref, _ = oracle.minibatch(rp, ci, init, 1, batch, law=law, weight=1.5, w_edge=we)
            with bl.Graph(rp, ci, we) as g:
                xy, st = g.run(init, algo=law, iters=1, batch=batch, weight=1.5, precision=bl.PREC_FP64)
            if law == 3:
                assert np.abs(xy - ref).max() <= 1e-10 * diameter(ref)
            else:
                assert np.array_equal(xy, ref) and st.energy == e_ref
