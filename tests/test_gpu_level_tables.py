"""Chunk descriptors of a level whose children differ much in size: one child keeps nearly all rows, so that its chunks exceed what its share of the
block's lanes writes, beside many children of one chunk; both partitions, against the fixed-point oracle."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import assert_tree_bits, setup_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,D,weights", [(400_003, 8, True), (400_003, 8, False), (2_300_001, 4, True), (1_100_001, 10, False), (30_001, 12, True)])
def test_one_child_keeps_the_rows(evt, N, D, weights):
    rng = np.random.default_rng(D)
    F, B = 18, 8
    x_bin = np.where(rng.random((F, N)) < 0.985, 1, rng.integers(2, B + 1, (F, N))).astype(np.uint8)
    y = (sum((x_bin[j] > 1) * 0.8**j for j in range(F)) + 0.1 * rng.random(N)).astype(np.float32)
    w = (0.5 + rng.random(N)).astype(np.float32) if weights else None
    h, o, op, gp, pred0, grad = setup_pair(evt, "mse", x_bin, y, w, np.zeros(1, np.float32), B, D, min_weight=0.0)
    orc.update_grads(op, pred0, y, grad)
    h.set_option("small_tree", 0)
    h.set_grads(grad)
    js = np.arange(1, F + 1, dtype=np.uint32)
    t, ids = h.grow_tree(js, gp), h.get_nidx()
    o.set_quant(grad, h.get_quant()[0])
    t_fx, ids_fx = o.grow_tree(grad, np.arange(N, dtype=np.uint32), js, mode=1)
    assert_tree_bits(t, t_fx)
    assert np.array_equal(ids, ids_fx)
    assert np.bincount(ids, minlength=2).max() > N // 2 and t.split.sum() > D  # the rows' last node, and others beside the way to it
    h.close()
    o.close()
