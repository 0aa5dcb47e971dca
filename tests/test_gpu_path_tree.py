"""A small tree in one launch (option "small_tree" = 4) against the histogram / search / partition kernels (= 0): trees, histograms, node ids, gradients and
predictions over free-running rounds, bit for bit, at the edges of what that kernel takes, and in turn with the other forms on one handle."""
import numpy as np
import pytest

from test_gpu_parity import assert_tree_bits, make_data

pytestmark = pytest.mark.gpu


def _assert_same(a, b):
    if isinstance(a, np.ndarray):
        assert a.tobytes() == b.tobytes()
    else:
        assert_tree_bits(a, b)


@pytest.mark.parametrize("N,F,B,D,loss,more", [
    (4, 1, 2, 2, "mse", {}),
    (5, 3, 16, 3, "mse", dict(weights=True)),
    (1023, 7, 64, 6, "logloss", dict(sub="drawn")),
    (1024, 10, 64, 6, "mse", {}),
    (1025, 16, 65, 5, "mse", dict(weights=True, sub="mask")),
    (2048, 17, 128, 4, "poisson", {}),
    (2049, 33, 129, 5, "mae", dict(sub="drawn")),
    (4099, 10, 64, 10, "mse", {}),                                    # 256 blocks, nodes of few rows and none
    (3001, 5, 255, 9, "logloss", dict(weights=True)),
    (1501, 64, 32, 5, "mse", {}),                                     # as many features as it takes
    (1200, 100, 16, 4, "gamma", dict(colsample=0.6)),                 # of more, sampled
    (6030, 4, 33, 4, "mse", dict(sub="drawn")),                       # as many rows as LDS holds, or nearly
    (4300, 3, 64, 7, "cred_var", {}),
    (2197, 9, 64, 6, "gaussian_mle", dict(weights=True, sub="mask")),
    (3001, 9, 100, 6, "mse", dict(cat=True, mono=True, sub="mask")),
    (2001, 9, 32, 6, "gaussian_mle", dict(cat=True, mono=True)),
    (2003, 6, 200, 5, "logistic_mle", dict(weights=True, cat=True)),
    (777, 6, 200, 4, "tweedie", dict(weights=True, cat=True, sub="drawn")),
    (999, 4, 64, 6, "mse", dict(sub="none")),                         # no row in the sample
])
def test_one_launch_a_tree_changes_nothing(evt, N, F, B, D, loss, more):
    rng = np.random.default_rng(N)
    x_bin, y, w, mu = make_data(N, N, F, B, loss, more.get("weights", False))
    ft = (rng.random(F) > 0.4).astype(np.uint8) if more.get("cat") else None
    mono = rng.integers(-1, 2, F).astype(np.int32) if more.get("mono") else None
    nfs = max(1, int(F * more.get("colsample", 1.0)))
    R = 5
    jss = [np.sort(rng.choice(F, nfs, replace=False)).astype(np.uint32) + 1 for _ in range(R)]
    masks = [rng.integers(0, 256, N, dtype=np.uint8) for _ in range(R)]
    gp = evt.make_params(eta=0.4, min_weight=0.0 if N < 10 else 2.0, L2=1.0)
    out = []
    # 9: the forms in turn, so that each finds what another has left
    for form in (4, 0, 9):
        for ahead in (0, 1):
            h = evt.Handle(N, F, B, len(mu), D, loss)
            h.set_option("grads_ahead", ahead)
            h.set_xbin(x_bin)
            h.set_feature_meta(ft, mono)
            h.set_target(y, w, mu)
            rec = []
            for r in range(R):
                h.set_option("small_tree", (4, 2, 4, 4, 0)[r] if form == 9 else form)
                h.update_grads()
                if more.get("sub") == "none":
                    with pytest.raises(evt.EvtError):
                        h.grow_tree(jss[r], gp, mask=np.full(N, 255, np.uint8), cond=140)
                elif more.get("sub") == "drawn":
                    h.draw_mask(r + 5)
                    h.grow_tree_begin_staged(jss[r], gp, 140)
                    rec.append(h.grow_tree_end())
                else:
                    rec.append(h.grow_tree(jss[r], gp, mask=masks[r] if more.get("sub") else None, cond=140))
                rec += [h.get_hist(), h.get_nidx()]
                if r != 1:  # with and without the predictions read between two rounds
                    rec.append(h.get_pred())
            h.update_grads()
            rec += [h.get_grads(), h.get_pred(), np.concatenate(h.get_quant())]
            h.close()
            out.append(rec)
    for rec in out:
        assert len(rec) == len(out[0])
        for a, b in zip(rec, out[2]):
            _assert_same(a, b)
    assert more.get("sub") == "none" or N < 10 or sum(int(t.split.sum()) for t in out[0] if not isinstance(t, np.ndarray)) > 0


@pytest.mark.parametrize("weights", [False, True])
def test_targets_gradients_and_bags_between_trees_of_one_launch(evt, weights):
    """New targets and weights, gradients from outside and several trees on the same gradients, between trees of one launch and others."""
    N, F, B, D = 2501, 8, 64, 5
    rng = np.random.default_rng(3)
    x_bin, y, w, mu = make_data(N, N, F, B, "mse", weights)
    js = np.arange(1, F + 1, dtype=np.uint32)
    gp = evt.make_params(eta=0.3, L2=1.0)
    bag = evt.make_params(eta=0.3, L2=1.0, bagging_size=2)
    out = []
    for forms in ([4] * 12, [0] * 12, [4, 0, 4, 4, 0, 2, 4, 3, 4, 4, 0, 4]):
        h = evt.Handle(N, F, B, 1, D, "mse")
        h.set_option("grads_ahead", 1)
        h.set_xbin(x_bin)
        h.set_target(y, w, mu)
        rec, it = [], iter(forms)

        def grow(params):
            h.set_option("small_tree", next(it))
            rec.extend([h.grow_tree(js, params), h.get_hist(), np.concatenate(h.get_quant()), h.get_nidx(), h.get_pred(), h.get_grads()])

        for _ in range(3):
            h.update_grads()
            grow(gp)
        h.update_grads()
        grow(bag)
        grow(bag)
        h.set_target(y * np.float32(2.0 ** -9), None if weights else (rng.random(N) * 0 + 1.5).astype(np.float32), mu * np.float32(2.0 ** -9))
        for _ in range(2):
            h.update_grads()
            grow(gp)
        h.set_grads(h.get_grads() * np.array([0.25, 0.25, 1.0], np.float32))
        grow(gp)
        for _ in range(4):
            h.update_grads()
            grow(gp)
        rec.append(h.get_grads())
        h.close()
        out.append(rec)
    for rec in out:
        for a, b in zip(rec, out[1]):
            _assert_same(a, b)
