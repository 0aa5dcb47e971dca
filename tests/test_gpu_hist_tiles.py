"""Column tiles of the conflict-free histogram kernel (option "hist_tile"): every width that a record's layout allows gives the fixed-point oracle's
tree and histograms, bit for bit, as does the width that the launch picks itself."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import assert_tree_bits, make_data, setup_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("loss,weights,K,N,F,B,D,n_js", [
    ("mse", False, None, 70_001, 100, 64, 5, 100),        # 7 features to a piece of 8 bytes: halves of 4 and of 3
    ("mse", True, None, 20_011, 65, 255, 4, 40),          # 5 to a piece: halves of 4 and of 1; fewer features than the record sampled
    ("logloss", False, None, 9_001, 92, 33, 4, 20),       # 6 to a piece, most features left out
    ("logloss", False, None, 65_537, 28, 128, 6, 28),     # 32-byte records
    ("logloss", True, None, 3_001, 17, 7, 4, 9),          # one feature in a record's second half, bins no multiple of 8
    ("mse", False, None, 5_003, 33, 100, 5, 33),          # 3 to a piece of 4 bytes
    ("gaussian_mle", False, None, 30_001, 50, 64, 5, 50),  # four channels, pieces of one byte
    ("gaussian_mle", True, None, 8_009, 64, 255, 4, 50),  # five channels of 255 bins: the 16-byte tile fits alone
    ("mlogloss", False, 7, 12_007, 30, 64, 4, 30),        # block layers
    ("mlogloss", True, 3, 6_001, 60, 255, 4, 30),         # block layers of 16-byte tiles only
    ("mse", False, None, 4_001, 120, 2, 2, 120),          # the fewest bins there are
    ("mse", True, None, 6_007, 300, 16, 4, 250),          # 320-byte records: the last tile is part padding
    ("gaussian_mle", False, None, 2_003, 1100, 16, 3, 900),
])
def test_every_tile_width_gives_the_same_tree(evt, loss, weights, K, N, F, B, D, n_js):
    x_bin, y, w, mu = make_data(3, N, F, B, loss, weights, K=K)
    h, o, op, gp, pred0, grad = setup_pair(evt, loss, x_bin, y, w, mu, B, D)
    orc.update_grads(op, pred0, y, grad)
    h.set_option("small_tree", 0)
    h.set_grads(grad)
    js = (np.sort(np.random.default_rng(N).choice(F, n_js, replace=False)) + 1).astype(np.uint32)
    gp.update_pred = 0
    trees, hists = [], []
    for tile, blocks in ((0, 256), (512, 256), (128, 256), (64, 256), (32, 256), (16, 256), (16, 3), (64, 31)):
        print("tile", tile, "blocks", blocks, flush=True)
        h.set_option("hist_tile", tile)
        h.set_option("hist_blocks", blocks)
        trees.append(h.grow_tree(js, gp))
        hists.append(h.get_hist())
    qb, _ = h.get_quant()
    o.set_quant(grad, qb)
    t_fx, _ = o.grow_tree(grad, np.arange(N, dtype=np.uint32), js, mode=1)
    for t, hist in zip(trees, hists):
        assert_tree_bits(t, t_fx)
        assert hist.tobytes() == hists[0].tobytes()
    assert t_fx.split.any()
    h.close()
    o.close()


@pytest.mark.parametrize("loss,weights,K,F,B", [("mse", False, None, 20, 16), ("mse", False, None, 100, 255), ("gaussian_mle", True, None, 33, 64)])
def test_shares_of_steps_and_of_iterations(evt, loss, weights, K, F, B):
    """Rows around the edges of a block's share, rounded up to steps (few spans, little to flush) and to whole iterations (many): the histograms
    of the generic kernel."""
    for N in (63, 64, 65, 1023, 1024, 1025, 4097, 31 * 1024 + 1, 131_073):
        x_bin, y, w, mu = make_data(N, N, F, B, loss, weights, K=K)
        h = evt.Handle(N, F, B, mu.shape[0], 3, loss)
        h.set_option("small_tree", 0)
        h.set_option("hist_in_scatter", 0)
        h.set_xbin(x_bin)
        h.set_target(y, w, mu)
        h.update_grads()
        gp = evt.make_params()
        gp.update_pred = 0
        js = np.arange(1, F + 1, dtype=np.uint32)
        got = []
        for variant, blocks in ((1, 256), (0, 256), (0, 31), (0, 2)):
            h.set_option("hist_variant", variant)
            h.set_option("hist_blocks", blocks)
            got.append((h.grow_tree(js, gp), h.get_hist()))
        h.close()
        for t, hist in got[1:]:
            assert_tree_bits(t, got[0][0])
            assert hist.tobytes() == got[0][1].tobytes()
