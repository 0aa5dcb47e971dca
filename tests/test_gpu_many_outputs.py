"""Kernels of any number of outputs at the edges of their split: gradients and their rows' maxima (bounds of 4, 8 and 16 classes), and the split search
with a wavefront per two outputs, against the fixed-point oracle and the two-launch form."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import assert_tree_bits, make_data, setup_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K", [(1, 2), (255, 4), (257, 5), (4_001, 8), (70_001, 9), (3_001, 16)])
def test_class_gradients_and_their_maxima(evt, N, K):
    x_bin, y, w, mu = make_data(K, N, 20, 16, "mlogloss", True, K=K)
    h = evt.Handle(N, 20, 16, K, 4, "mlogloss")
    h.set_option("small_tree", 0)
    h.set_xbin(x_bin)
    h.set_target(y, w, mu)
    js = np.arange(1, 21, dtype=np.uint32)
    for _ in range(3):
        h.update_grads()  # from the second round on with the last tree's leaf values added on the way
        g, p = h.get_grads(), h.get_pred().astype(np.float64)
        e = np.exp(p)
        prob = e / e.sum(1, keepdims=True)
        want = (prob - (y[:, None] == np.arange(1, K + 1))) * w[:, None]
        bound = (K + 4) * 2.0**-23 * 1.5  # exponentials to an ulp, K sums, a quotient and a product; weights below 1.5
        assert np.abs(g[:, :K] - want).max() <= bound
        assert np.abs(g[:, K:2 * K] - prob * (1 - prob) * w[:, None]).max() <= 2 * bound
        h.grow_tree(js, evt.make_params(eta=0.3, min_weight=0.0))
        _, qexp = h.get_quant()  # of the tree's gradients
        big = np.abs(g).max(0)
        assert np.array_equal(qexp, np.where(big > 0, np.frexp(big)[1], 0))
    h.close()


@pytest.mark.parametrize("N,F,B,D,K,n_js,tt,cat", [
    (3_001, 3, 100, 6, 2, 3, "binary", False),     # two bins to a lane, one wavefront to a feature
    (5_003, 9, 255, 5, 9, 7, "binary", True),      # four, and an odd number of outputs
    (2_001, 5, 255, 4, 16, 5, "binary", False),    # the largest block
    (40, 4, 64, 6, 3, 4, "binary", True),          # empty nodes and leaves at every level
    (4_001, 6, 65, 5, 5, 6, "oblivious", False),
    (6_001, 258, 16, 8, 9, 256, "binary", True),    # from 32 nodes of 256 features on two wavefronts take the pairs of 9 to 14 outputs in turn
    (5_001, 129, 70, 8, 14, 128, "oblivious", False),
    (3_001, 256, 129, 7, 10, 256, "binary", False),
])
def test_search_of_many_outputs(evt, N, F, B, D, K, n_js, tt, cat):
    rng = np.random.default_rng(N)
    ft = (rng.random(F) > 0.5).astype(np.uint8) if cat else None
    x_bin, y, w, mu = make_data(3, N, F, B, "mlogloss", N % 2 == 0, K=K)
    h, o, op, gp, pred0, grad = setup_pair(evt, "mlogloss", x_bin, y, w, mu, B, D, tt, feattypes=ft, min_weight=0.0)
    orc.update_grads(op, pred0, y, grad)
    h.set_option("small_tree", 0)
    gp.update_pred = 0
    js = (np.sort(rng.choice(F, n_js, replace=False)) + 1).astype(np.uint32)
    h.set_grads(grad)
    got = []
    for fused in (1, 0, 1):
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
