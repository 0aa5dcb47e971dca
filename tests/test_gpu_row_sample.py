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


@pytest.mark.parametrize("loss,weights,N", [("mse", False, 8_191), ("mse", False, 8_193), ("logloss", True, 16_389), ("gaussian_mle", False, 1_048_577),
                                            ("mse", False, 2_100_003), ("mse", True, 2_100_003)])
def test_drawn_rows_beside_the_quantisation(evt, loss, weights, N):
    """The mask drawn on the way, its last bytes and blocks partly filled, while blocks of the same kernel quantise the device's own gradients."""
    F, B, D = 6, 16, 3
    x_bin, y, w, mu = make_data(N, N, F, B, loss, weights)
    h, o, op, gp, pred0, grad = setup_pair(evt, loss, x_bin, y, w, mu, B, D)
    h.set_option("small_tree", 0)
    js = np.arange(1, F + 1, dtype=np.uint32)
    for k, cond in enumerate((127, 204, 1)):
        seed = 1_000_003 * N + k
        h.update_grads()
        grad = h.get_grads()
        h.draw_mask(seed)
        h.grow_tree_begin_staged(js, gp, cond)
        t = h.grow_tree_end()
        rows = np.flatnonzero(evt.splitmix_mask(seed, N) <= cond).astype(np.uint32)
        o.set_quant(grad, h.get_quant()[0])
        t_fx, nidx = o.grow_tree(grad, rows, js, mode=1)
        assert_tree_bits(t, t_fx)
        got, want = h.get_nidx(), np.zeros(N, np.uint32)
        want[rows] = np.asarray(nidx)[rows]
        assert np.array_equal(got, want)
    h.close()
    o.close()
