"""The widest chunks of the one-pass partition, which the root and the first levels of millions of rows take, against the count and scatter passes: trees, histograms,
node ids and predictions, bit for bit, with chunks that end inside a wavefront's rows."""
import numpy as np
import pytest

from test_gpu_parity import assert_tree_bits, make_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,more", [
    (2_097_153, {}),                                # the first size that takes chunks of 16 384 rows at the root
    (4_194_304 + 16_385, dict(cat=True, planes=0)),  # ... and at both nodes below it; bin bytes decide
    (3_000_017, dict(sub=True)),
])
def test_wide_chunks_change_nothing(evt, N, more):
    F, B, D = 17, 8, 5
    rng = np.random.default_rng(N)
    x_bin, y, _, mu = make_data(N, N, F, B, "mse", False)
    ft = (rng.random(F) > 0.5).astype(np.uint8) if more.get("cat") else None
    js = np.arange(1, F + 1, dtype=np.uint32)
    gp = evt.make_params(eta=0.4, L2=1.0)
    mask = rng.integers(0, 256, N, dtype=np.uint8) if more.get("sub") else None
    out = []
    for one in (1, 0):
        h = evt.Handle(N, F, B, 1, D, "mse")
        h.set_option("part_one_pass", one)
        h.set_option("bit_planes", more.get("planes", 1))
        h.set_xbin(x_bin)
        h.set_feature_meta(ft, None)
        h.set_target(y, None, mu)
        h.update_grads()
        t = h.grow_tree(js, gp, mask=mask, cond=250 if more.get("sub") else 255)
        out.append((t, h.get_hist(), h.get_nidx(), h.get_pred()))
        h.close()
    a, b = out
    assert_tree_bits(a[0], b[0])
    for u, v in zip(a[1:], b[1:]):
        assert u.tobytes() == v.tobytes()
    assert a[0].split.sum() >= 7
