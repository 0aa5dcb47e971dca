"""An oblivious level in one launch (option "scan_fused" = 1) against three (= 0) and the fixed-point oracle, at the edges of the rule that chooses it."""
import numpy as np
import pytest

from oracle import oracle as orc
from test_gpu_parity import assert_tree_bits, make_data, setup_pair

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("loss,weights,N,F,B,D,n_js,more", [
    ("mse", False, 5_001, 1, 4, 3, 1, {}),                               # one block, the fewest bins
    ("mse", True, 5_001, 6, 3, 4, 6, {}),                                # fewer: three launches
    ("mse", False, 20_001, 70, 64, 8, 65, {}),                           # 32 nodes in one, 64 in three; 65 candidates
    ("mse", False, 20_001, 20, 65, 7, 20, {}),                           # two bins to a lane
    ("logloss", True, 20_001, 20, 128, 7, 20, dict(cat=True)),
    ("logloss", False, 20_001, 20, 255, 6, 17, dict(cat=True, mono=True)),
    ("gaussian_mle", False, 20_001, 18, 64, 7, 18, {}),                  # 32 nodes, the last of them with leaves
    ("gaussian_mle", True, 9_001, 18, 255, 5, 18, dict(cat=True)),       # the largest block's registers
    ("gaussian_mle", False, 9_001, 18, 200, 6, 18, {}),                  # 8 nodes in one, 16 in three
    ("mse", False, 300, 20, 32, 7, 20, dict(min_weight=20.0)),           # levels without a split
    ("mse", False, 5_001, 20, 32, 4, 20, dict(gamma=1e9)),               # the root is a leaf
    ("mae", True, 5_001, 20, 32, 5, 20, {}),
    # 129 to 192 bins are three pieces of 64 but four bins to a lane: two channels take 32 nodes in one launch, and 64 in three
    ("mse", False, 20_001, 20, 129, 7, 20, {}),
    ("mse", True, 20_001, 20, 160, 8, 17, dict(cat=True, mono=True)),
    ("mae", False, 20_001, 66, 192, 8, 66, {}),
    ("mse", False, 20_001, 20, 193, 7, 20, {}),                          # four pieces: 16 nodes in one, 32 in three
    ("logloss", False, 20_001, 20, 160, 7, 20, {}),
    ("gaussian_mle", True, 20_001, 18, 160, 6, 18, {}),
])
def test_one_launch_decides_the_level(evt, loss, weights, N, F, B, D, n_js, more):
    more = dict(more)
    rng = np.random.default_rng(N + B)
    ft = (rng.random(F) > 0.4).astype(np.uint8) if more.pop("cat", False) else None
    mono = rng.integers(-1, 2, F).astype(np.int32) if more.pop("mono", False) else None
    x_bin, y, w, mu = make_data(5, N, F, B, loss, weights)
    h, o, op, gp, pred0, grad = setup_pair(evt, loss, x_bin, y, w, mu, B, D, "oblivious", feattypes=ft, mono=mono, **more)
    orc.update_grads(op, pred0, y, grad)
    h.set_option("small_tree", 0)
    gp.update_pred = 0
    jss = [(np.sort(rng.choice(F, n_js, replace=False)) + 1).astype(np.uint32) for _ in range(2)]
    for js in jss:
        h.set_grads(grad)
        got = []
        for fused in (1, 0, 1, 1):  # a level's blocks are counted, and the count has to be back at zero
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
