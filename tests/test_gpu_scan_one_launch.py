"""The split search whose last block decides the node (option "scan_fused" = 1, more than 16 sampled features) against the fixed-point oracle and the two
kernels (= 0), tree after tree on one handle: a node's blocks are counted, and the count has to be back at zero."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import assert_tree_bits, make_data, setup_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("loss,weights,N,F,B,D,n_js,more", [
    ("mse", False, 9_001, 17, 64, 7, 17, {}),                                # five groups, the last of one feature
    ("mse", True, 4_003, 260, 16, 5, 256, {}),                               # 64 groups: one candidate to a lane
    ("mse", False, 4_003, 300, 16, 5, 257, {}),                              # 65
    ("logloss", False, 20_011, 28, 255, 9, 28, dict(min_weight=0.0)),        # hundreds of nodes, some of them empty
    ("gaussian_mle", True, 9_001, 40, 100, 6, 33, {}),
    ("mse", False, 5_001, 30, 32, 2, 30, {}),                                # the root alone splits; its children are leaves
    ("mse", False, 5_001, 30, 32, 5, 30, dict(gamma=1e9)),                   # no candidate is good enough
    ("logloss", True, 900, 20, 32, 4, 20, dict(min_weight=1e6)),             # there is no candidate
    ("mse", True, 6_001, 50, 64, 6, 50, dict(cat=True, mono=True)),
    ("mlogloss", False, 9_001, 3, 64, 6, 3, dict(K=7)),                      # any number of outputs: one block to a node
    ("mlogloss", True, 9_001, 30, 255, 7, 26, dict(K=3, cat=True)),
    ("mlogloss", False, 3_001, 280, 16, 4, 261, dict(K=5)),
    ("mlogloss", False, 3_001, 20, 16, 4, 20, dict(K=16, gamma=1e9)),
])
def test_last_block_decides(evt, loss, weights, N, F, B, D, n_js, more):
    more = dict(more)
    rng = np.random.default_rng(N)
    ft = (rng.random(F) > 0.4).astype(np.uint8) if more.pop("cat", False) else None
    mono = rng.integers(-1, 2, F).astype(np.int32) if more.pop("mono", False) else None
    x_bin, y, w, mu = make_data(5, N, F, B, loss, weights, K=more.pop("K", None))
    h, o, op, gp, pred0, grad = setup_pair(evt, loss, x_bin, y, w, mu, B, D, feattypes=ft, mono=mono, **more)
    orc.update_grads(op, pred0, y, grad)
    h.set_option("small_tree", 0)
    gp.update_pred = 0
    jss = [(np.sort(rng.choice(F, n_js, replace=False)) + 1).astype(np.uint32) for _ in range(2)]
    for js in jss:
        h.set_grads(grad)
        got = []
        for fused in (1, 0, 1, 1):
            h.set_option("scan_fused", fused)
            got.append((h.grow_tree(js, gp), h.get_hist(), h.get_nidx()))
        qb, _ = h.get_quant()
        o.set_quant(grad, qb)
        t_fx, nidx = o.grow_tree(grad, np.arange(N, dtype=np.uint32), js, mode=1)
        for t, hist, ids in got:
            assert_tree_bits(t, t_fx)
            assert hist.tobytes() == got[0][1].tobytes()
            assert np.array_equal(ids, nidx)
    h.close()
    o.close()
