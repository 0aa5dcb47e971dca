"""Records that lie further than 32 bits hold from the first one: the histograms and the tree of a sample of the last features are those of a handle
that has these features alone."""
import numpy as np
import pytest

from test_gpu_parity import assert_tree_bits, make_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("loss", ["mse", "gaussian_mle"])
def test_records_past_four_gigabytes(evt, loss):
    N, F, B, D = 1_080_001, 4000, 8, 3
    assert N * F > 1 << 32  # a byte a feature
    x8, y, w, mu = make_data(5, N, 8, B, loss, False)
    x8 = np.ascontiguousarray(x8)
    got = []
    for x in (np.tile(x8, (F // 8, 1)), x8):
        feats = x.shape[0]
        print("features", feats, flush=True)
        h = evt.Handle(N, feats, B, mu.shape[0], D, loss)
        h.set_option("small_tree", 0)
        h.set_xbin(x)
        h.set_feature_meta(None, None)
        h.set_target(y, w, mu)
        h.update_grads()
        js = np.arange(feats - 7, feats + 1, dtype=np.uint32)
        tree = h.grow_tree(js, evt.make_params())
        tree.feat[tree.feat > 0] -= feats - 8
        got.append((tree, np.ascontiguousarray(h.get_hist()[:, feats - 8:])))
        h.close()
    assert got[0][0].split.any()
    assert_tree_bits(got[0][0], got[1][0])
    assert got[0][1].tobytes() == got[1][1].tobytes()


def test_half_the_features_past_four_gigabytes(evt):
    """Half of the features, the last ones, which repeat eight: the kernel without a test per feature."""
    N, F, B, D = 1_080_001, 4000, 8, 3
    x8, y, w, mu = make_data(6, N, 8, B, "mse", True)
    x8 = np.ascontiguousarray(x8)
    got = []
    for x, n_js in ((np.tile(x8, (F // 8, 1)), F // 2), (x8, 8)):
        feats = x.shape[0]
        print("features", feats, flush=True)
        h = evt.Handle(N, feats, B, 1, D, "mse")
        h.set_option("small_tree", 0)
        h.set_xbin(x)
        h.set_target(y, w, mu)
        h.update_grads()
        tree = h.grow_tree(np.arange(feats - n_js + 1, feats + 1, dtype=np.uint32), evt.make_params())
        tree.feat[tree.feat > 0] -= feats - n_js
        got.append((tree, np.ascontiguousarray(h.get_hist()[:, feats - n_js:])))
        h.close()
    assert got[0][0].split.any()
    assert_tree_bits(got[0][0], got[1][0])
    for f in range(0, F // 2, 8):
        assert got[0][1][:, f:f + 8].tobytes() == got[1][1].tobytes()
