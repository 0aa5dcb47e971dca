"""Trees of either form on the same gradients: the words that a tree of few rows' kernels read in planes are made again side by side for the others, and
back, and every tree is the fixed-point oracle's, at each number of channels (one: planes alone; odd ones: padded rows)."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import assert_tree_bits, make_data, setup_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("loss,weights,K,N,F", [
    ("mse", False, None, 2_003, 20), ("mse", True, None, 2_003, 20), ("logloss", False, None, 1_001, 17), ("logloss", True, None, 1_001, 9),
    ("gaussian_mle", False, None, 4_003, 33), ("gaussian_mle", True, None, 777, 33), ("mlogloss", False, 3, 1_501, 12), ("mlogloss", True, 8, 1_501, 30),
    ("gaussian_mle", True, None, 60_013, 20), ("mse", True, None, 300_007, 8), ("mlogloss", True, 4, 40_009, 6),
])
def test_layouts_change_between_trees(evt, loss, weights, K, N, F):
    B = 32
    x_bin, y, w, mu = make_data(N, N, F, B, loss, weights, K=K)
    h, o, op, gp, pred0, grad = setup_pair(evt, loss, x_bin, y, w, mu, B, 4)
    orc.update_grads(op, pred0, y, grad)
    h.set_grads(grad)
    js = np.arange(1, F + 1, dtype=np.uint32)
    gp.update_pred = 0
    trees = []
    for form in (0, 2, 0, 0, 3, 2, 0):
        h.set_option("small_tree", form)
        trees.append(h.grow_tree(js, gp))
    o.set_quant(grad, h.get_quant()[0])
    t_fx, _ = o.grow_tree(grad, np.arange(N, dtype=np.uint32), js, mode=1)
    assert t_fx.split.any()
    for t in trees:
        assert_tree_bits(t, t_fx)
    for first in (2, 3, 0):  # the words made by the root's kernel of a small tree, or beside the other form's set-up, of the device's own gradients
        h.update_grads()
        trees = []
        for form in (first, 0, 3):
            h.set_option("small_tree", form)
            trees.append(h.grow_tree(js, gp))
        own = h.get_grads()
        o.set_quant(own, h.get_quant()[0])
        t_fx, _ = o.grow_tree(own, np.arange(N, dtype=np.uint32), js, mode=1)
        for t in trees:
            assert_tree_bits(t, t_fx)
    h.close()
    o.close()
