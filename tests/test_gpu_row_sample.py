"""Row samples in one kernel: around the edges of its blocks of 8192 rows, with masks that keep none of a block, all of it or single rows, the tree and its rows are
those of the oracle on the rows kept, tree after tree on one handle."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import assert_tree_bits, make_data, setup_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [4, 31, 32, 33, 8191, 8192, 8193, 16_385, 70_001])
@pytest.mark.parametrize("loss", ["mse", "logloss"])
def test_sampled_rows(evt, N, loss):
    F, B = 20, 16
    x_bin, y, w, mu = make_data(N, N, F, B, loss, False)
    h, o, op, gp, pred0, grad = setup_pair(evt, loss, x_bin, y, w, mu, B, 4)
    orc.update_grads(op, pred0, y, grad)
    h.set_option("small_tree", 0)
    h.set_option("record_nidx", 1)
    h.set_grads(grad)
    js = np.arange(1, F + 1, dtype=np.uint32)
    gp.update_pred = 0
    rng = np.random.default_rng(N)
    masks = [rng.integers(0, 256, N).astype(np.uint8), np.where(np.arange(N) // 8192 % 2, 255, 0).astype(np.uint8),
             np.where(np.arange(N) == N - 1, 0, 255).astype(np.uint8), rng.integers(0, 256, N).astype(np.uint8)]
    for mask in masks:
        rows = np.flatnonzero(mask <= 127).astype(np.uint32)
        if rows.size == 0:
            with pytest.raises(evt.EvtError, match="no subsample"):
                h.grow_tree(js, gp, mask=mask, cond=127)
            continue
        t = h.grow_tree(js, gp, mask=mask, cond=127)
        o.set_quant(grad, h.get_quant()[0])
        t_fx, nidx = o.grow_tree(grad, rows, js, mode=1)
        assert_tree_bits(t, t_fx)
        got = h.get_nidx()
        assert not got[mask > 127].any() and np.array_equal(got[rows], np.asarray(nidx)[rows])
    h.close()
    o.close()


@pytest.mark.parametrize("N", [1_003, 8_193, 30_011])
def test_few_rows_of_a_large_root_slice(evt, N):
    """Blocks of their own clear the root's slice: 306,000 words, which the trees before have filled."""
    F, B, K = 80, 255, 7
    x_bin, y, w, mu = make_data(N, N, F, B, "mlogloss", True, K=K)
    h, o, op, gp, pred0, grad = setup_pair(evt, "mlogloss", x_bin, y, w, mu, B, 2)
    orc.update_grads(op, pred0, y, grad)
    h.set_option("small_tree", 0)
    h.set_grads(grad)
    js = np.arange(1, F + 1, dtype=np.uint32)
    gp.update_pred = 0
    o.set_quant(grad, h.get_quant()[0])
    rng = np.random.default_rng(N)
    for cond in (127, 255, 20, 200):
        mask = rng.integers(0, 256, N).astype(np.uint8)
        t = h.grow_tree(js, gp, mask=mask, cond=cond)
        t_fx, _ = o.grow_tree(grad, np.flatnonzero(mask <= cond).astype(np.uint32), js, mode=1)
        assert_tree_bits(t, t_fx)
        assert t.split.any()
    h.close()
    o.close()
