"""Five accumulator channels around the number of bins from which the narrowest histogram tile takes all of a CU's LDS: the oracle's trees and the
generic kernel's histograms."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import assert_tree_bits, make_data, setup_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,F,B,n_js", [(3_001, 17, 204, 17), (3_001, 17, 205, 9), (70_001, 40, 255, 40), (9_001, 100, 255, 30), (2_003, 700, 230, 700)])
def test_five_channels_of_many_bins(evt, N, F, B, n_js):
    x_bin, y, w, mu = make_data(B, N, F, B, "gaussian_mle", True)
    h, o, op, gp, pred0, grad = setup_pair(evt, "gaussian_mle", x_bin, y, w, mu, B, 4)
    orc.update_grads(op, pred0, y, grad)
    h.set_option("small_tree", 0)
    h.set_grads(grad)
    js = (np.sort(np.random.default_rng(N).choice(F, n_js, replace=False)) + 1).astype(np.uint32)
    gp.update_pred = 0
    got = []
    for variant, blocks in ((2, 256), (1, 256), (2, 5)):
        h.set_option("hist_variant", variant)
        h.set_option("hist_blocks", blocks)
        got.append((h.grow_tree(js, gp), h.get_hist()))
    o.set_quant(grad, h.get_quant()[0])
    t_fx, _ = o.grow_tree(grad, np.arange(N, dtype=np.uint32), js, mode=1)
    assert t_fx.split.any()
    for t, hist in got:
        assert_tree_bits(t, t_fx)
        assert hist.tobytes() == got[0][1].tobytes()
    h.close()
    o.close()
