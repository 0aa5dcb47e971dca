"""The partition of a level in one kernel (option "part_one_pass" = 1, unit weights) against the count and scatter passes (= 0): trees, histograms,
node ids and predictions over free-running rounds, bit for bit, on both sides of a chunk's edges and of each chunk size."""
import numpy as np
import pytest

from test_gpu_parity import assert_tree_bits, make_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,F,B,D,loss,more", [
    (1, 17, 4, 3, "mse", {}),
    (2_047, 17, 16, 4, "mse", {}),
    (2_049, 17, 16, 11, "mse", {}),                                   # nodes of few rows, leaves at every level
    (6_145, 20, 32, 6, "logloss", dict(cat=True)),                    # bin bytes decide beside bit planes
    (9_001, 20, 32, 6, "gaussian_mle", dict(planes=0)),
    (262_143, 17, 8, 5, "mse", {}),                                   # the root's chunks: 2048 rows
    (262_145 + 2_048, 17, 8, 5, "mse", {}),                           # 4096
    (530_001, 17, 8, 4, "mse", dict(defer=0)),                        # 8192, then 4096; leaf values added on the way
    (1_050_001, 17, 8, 4, "logloss", dict(sub=True)),                 # chunks by the sample's size
    (30_011, 18, 16, 5, "mlogloss", dict(K=5)),
    (30_011, 18, 16, 6, "mse", dict(tt="oblivious")),
    (70_001, 17, 8, 13, "mse", {}),                                   # cursors past the first thousand
    # every node of the level of 8192 is split: more chunks than the 4096 blocks of a launch, each of which takes several in turn
    (100_003, 17, 2, 16, "mse", dict(L2=0.0)),
    (200_003, 18, 2, 16, "mse", dict(L2=0.0, sub=True)),
])
def test_one_pass_changes_nothing(evt, N, F, B, D, loss, more):
    rng = np.random.default_rng(N)
    x_bin, y, _, mu = make_data(N, N, F, B, loss, False, K=more.get("K"))
    ft = (rng.random(F) > 0.5).astype(np.uint8) if more.get("cat") else None
    js = np.arange(1, F + 1, dtype=np.uint32)
    gp = evt.make_params(eta=0.4, L2=more.get("L2", 1.0), min_weight=0.0 if N < 3_000 else 1.0)
    out = []
    for one in (1, 0):
        h = evt.Handle(N, F, B, len(mu), D, loss, more.get("tt", "binary"))
        h.set_option("small_tree", 0)
        h.set_option("part_one_pass", one)
        h.set_option("bit_planes", more.get("planes", 1))
        h.set_option("defer_pred", more.get("defer", 1))
        h.set_xbin(x_bin)
        h.set_feature_meta(ft, None)
        h.set_target(y, None, mu)
        rec = []
        for r in range(3):
            h.update_grads()
            mask = np.random.default_rng(r).integers(0, 256, N, dtype=np.uint8) if more.get("sub") else None
            t = h.grow_tree(js, gp, mask=mask, cond=180 if more.get("sub") else 255)
            rec.append((t, h.get_hist(), h.get_nidx(), h.get_pred()))
        h.close()
        out.append(rec)
    for a, b in zip(*out):
        assert_tree_bits(a[0], b[0])
        for u, v in zip(a[1:], b[1:]):
            assert u.tobytes() == v.tobytes()
    assert N == 1 or out[0][0][0].split.sum() >= 1
    if D == 16:
        assert (out[0][0][0].split[2**13 - 1 : 2**14 - 1]).sum() > 5_000
