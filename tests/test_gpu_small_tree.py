"""One and two kernels per level (option "small_tree" = 2 and 3) against the histogram / search / partition kernels (= 0): trees, histograms, node ids,
gradients and predictions over free-running rounds, bit for bit, at the edges of what that path takes."""
import numpy as np
import pytest

from test_gpu_parity import assert_tree_bits, make_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,F,B,D,loss,more", [
    (4, 1, 2, 2, "mse", {}),
    (5, 3, 16, 3, "mse", dict(weights=True)),
    (1023, 7, 64, 6, "logloss", dict(sub="drawn")),
    (4099, 10, 64, 10, "mse", {}),                                   # 256 nodes, several to a wavefront
    (3001, 5, 255, 9, "logloss", dict(weights=True)),                # more nodes than LDS histograms: several passes over the rows
    (8197, 17, 129, 5, "gaussian_mle", dict(weights=True, sub="mask")),
    (65_535, 4, 33, 4, "mse", dict(sub="drawn")),
    (2002, 256, 8, 5, "mse", {}),
    (2500, 300, 8, 4, "poisson", dict(colsample=0.4)),
    (1500, 64, 8, 5, "mse", {}),                                      # a candidate to a lane, and one more
    (1500, 65, 8, 5, "gaussian_mle", dict(weights=True)),
    (1700, 193, 8, 7, "logloss", dict(oblivious=True, cat=True)),
    (1300, 129, 8, 5, "mlogloss", dict(K=3)),                         # two blocks each are more than the chip has units: searched apart
    (1300, 128, 8, 5, "mse", dict(oblivious=True)),
    (6001, 9, 32, 6, "gaussian_mle", dict(cat=True, mono=True)),
    (6001, 9, 100, 6, "mse", dict(cat=True, mono=True, sub="mask")),
    (5003, 12, 64, 7, "gaussian_mle", dict(oblivious=True)),
    (777, 6, 200, 4, "logloss", dict(oblivious=True, weights=True, cat=True, sub="drawn")),
    (4001, 8, 32, 5, "mlogloss", dict(K=7)),
    (2047, 8, 200, 6, "mlogloss", dict(K=3, weights=True, sub="mask", cat=True)),
    (1500, 5, 64, 4, "mlogloss", dict(K=16, oblivious=True)),
    (1200, 6, 64, 5, "mlogloss", dict(K=2)),
    (150_001, 3, 64, 6, "mse", dict(sub="drawn")),                   # more rows than one block per feature takes
    (70_001, 12, 40, 5, "gaussian_mle", dict(oblivious=True, weights=True)),
    # levels of shared rows on either side of the line where their searches take a kernel of their own
    (3001, 5, 255, 8, "gaussian_mle", dict(oblivious=True, weights=True)),
    (4001, 6, 255, 5, "gaussian_mle", dict(sub="mask")),
    (5001, 4, 128, 7, "gaussian_mle", {}),
    (6007, 3, 200, 8, "mse", dict(oblivious=True)),
    (3011, 4, 224, 7, "mse", dict(oblivious=True)),                  # 16 nodes of 448 words are the last that stay
    (3011, 4, 225, 7, "mse", dict(oblivious=True, weights=True)),
    (7001, 3, 160, 7, "mse", dict(weights=True)),                    # two nodes of 320 words are the last that stay
    (3001, 5, 64, 6, "mse", {}),                                      # eight nodes are 1024 words: apart; of 63 bins they stay
    (3001, 5, 63, 6, "mse", {}),
    (5001, 5, 192, 6, "logloss", dict(weights=True)),                # three channels, four bins to a lane: searched apart from the root on
    (5001, 4, 160, 6, "cred_var", dict(oblivious=True)),
    (5001, 4, 128, 6, "poisson", dict(oblivious=True, sub="drawn")),
    (2003, 4, 255, 5, "mlogloss", dict(K=16)),
    (2503, 4, 255, 6, "mlogloss", dict(K=5, oblivious=True)),
])
def test_one_kernel_per_level_changes_nothing(evt, N, F, B, D, loss, more):
    rng = np.random.default_rng(N)
    K = more.get("K")
    if K:
        x_bin = rng.integers(1, B + 1, size=(F, N), dtype=np.uint8)
        y = (1 + (x_bin[0].astype(int) * K // (B + 1) + rng.integers(0, 2, N)) % K).astype(np.float32)
        mu = np.zeros(K, np.float32)
        w = (rng.random(N) + 0.5).astype(np.float32) if more.get("weights") else None
    else:
        x_bin, y, w, mu = make_data(N, N, F, B, loss, more.get("weights", False))
    ft = (rng.random(F) > 0.4).astype(np.uint8) if more.get("cat") else None
    mono = rng.integers(-1, 2, F).astype(np.int32) if more.get("mono") else None
    nfs = max(1, int(F * more.get("colsample", 1.0)))
    R = 4
    jss = [np.sort(rng.choice(F, nfs, replace=False)).astype(np.uint32) + 1 for _ in range(R)]
    masks = [rng.integers(0, 256, N, dtype=np.uint8) for _ in range(R)]
    gp = evt.make_params(eta=0.4, min_weight=0.0 if N < 10 else 2.0, L2=1.0)
    out = []
    for small in (2, 3, 0):
        h = evt.Handle(N, F, B, len(mu), D, loss, "oblivious" if more.get("oblivious") else "binary")
        h.set_option("small_tree", small)
        h.set_xbin(x_bin)
        h.set_feature_meta(ft, mono)
        h.set_target(y, w, mu)
        rec = []
        for r in range(R):
            h.update_grads()
            if more.get("sub") == "drawn":
                h.draw_mask(r + 5)
                h.grow_tree_begin_staged(jss[r], gp, 140)
                rec.append(h.grow_tree_end())
            else:
                rec.append(h.grow_tree(jss[r], gp, mask=masks[r] if more.get("sub") else None, cond=140))
            rec += [h.get_hist(), h.get_nidx()]
            if r != 1:  # with and without the predictions read between two rounds
                rec.append(h.get_pred())
        h.update_grads()
        rec += [h.get_grads(), h.get_pred()]
        h.close()
        out.append(rec)
    splits = 0
    for a, a2, b in zip(*out):
        if isinstance(a, np.ndarray):
            assert a.tobytes() == b.tobytes() and a2.tobytes() == b.tobytes()
        else:
            assert_tree_bits(a, b)
            assert_tree_bits(a2, b)
            splits += int(a.split.sum())
    assert splits > 0 or N < 10


@pytest.mark.parametrize("N,B,loss,K", [(1030, 64, "mse", 1), (2501, 200, "logloss", 1), (1999, 33, "gaussian_mle", 2), (1500, 40, "mlogloss", 7),
                                        (63_000, 64, "mlogloss", 3), (63_001, 33, "mlogloss", 2)])  # 42 blocks a feature: quantised by the root, and ahead of it
def test_gradients_quantised_by_the_tree_or_not(evt, N, B, loss, K):
    """The root's kernel quantises what evt_update_grads left; whatever comes in between (a second update, other targets, gradients from outside,
    the other kernels, a second tree on the same gradients) sees what k_quantize would have left: same tables, trees and histograms."""
    F, D = 6, 4
    rng = np.random.default_rng(N)
    x_bin = rng.integers(1, B + 1, size=(F, N), dtype=np.uint8)
    if loss == "mlogloss":
        y, mu = (1 + (x_bin[0].astype(int) + rng.integers(0, 3, N)) % K).astype(np.float32), np.zeros(K, np.float32)
    else:
        _, y, _, mu = make_data(N, N, F, B, loss, False)
    small_y = y if loss in ("mlogloss", "logloss") else y * np.float32(2.0 ** -9)  # smaller maxima: none may be left of the first targets
    small_mu = mu if small_y is y else mu * np.float32(2.0 ** -9)
    w = (rng.random(N) + 0.5).astype(np.float32)
    js = np.arange(1, F + 1, dtype=np.uint32)
    gp = evt.make_params(eta=0.3, L2=1.0)
    keep = evt.make_params(eta=0.3, L2=1.0, update_pred=0, bagging_size=2)
    out = []
    for small in (2, 3, 0):
        h = evt.Handle(N, F, B, len(mu), D, loss)
        h.set_option("small_tree", small)
        h.set_xbin(x_bin)
        rec = []

        def note():
            rec.extend([h.get_hist(), np.concatenate(h.get_quant()), h.get_pred(), h.get_grads()])

        h.set_target(y, None, mu)
        h.update_grads()
        h.update_grads()
        rec.append(np.concatenate(h.get_quant()))  # before any tree
        rec.append(h.grow_tree(js, gp))
        note()
        h.update_grads()
        h.set_target(small_y, w, small_mu)  # other channels, smaller gradients
        h.update_grads()
        rec.append(h.grow_tree(js, keep))
        rec.append(h.grow_tree(js, keep))  # on the same gradients
        note()
        h.update_grads()
        h.set_option("small_tree", 0)
        rec.append(h.grow_tree(js, gp))
        h.set_option("small_tree", small)
        note()
        h.update_grads()
        h.set_grads(h.get_grads() * np.float32(0.25))
        rec.append(h.grow_tree(js, gp))
        note()
        h.close()
        out.append(rec)
    splits = 0
    for a, a2, b in zip(*out):
        if isinstance(a, np.ndarray):
            assert a.tobytes() == b.tobytes() and a2.tobytes() == b.tobytes()
        else:
            assert_tree_bits(a, b)
            assert_tree_bits(a2, b)
            splits += int(a.split.sum())
    assert splits > 0


@pytest.mark.parametrize("N,D,loss,more", [
    (4, 2, "mse", {}),
    (1025, 3, "mse", dict(weights=True, sub=True)),
    (2049, 5, "logloss", {}),                          # a last block of one row
    (1024, 4, "gaussian_mle", dict(weights=True)),
    (3000, 6, "gaussian_mle", dict(oblivious=True)),
    (1999, 4, "logistic_mle", dict(sub=True)),
    (1500, 4, "poisson", {}),
    (1500, 4, "gamma", dict(weights=True)),
    (1500, 4, "tweedie", {}),
    (1500, 4, "mae", dict(weights=True)),
    (1500, 4, "cred_var", {}),
    (1500, 4, "cred_std", dict(sub=True)),
    (1500, 4, "mlogloss", {}),                         # several outputs: the gradient kernels of their own
    (262_145, 4, "mse", dict(weights=True)),           # one row more than the last kernel's blocks take at once
    (530_001, 3, "gaussian_mle", {}),
    (530_001, 4, "logloss", dict(sub=True, weights=True)),  # the walk over all rows behind a sampled tree: wide blocks
    (2_097_153, 3, "mse", dict(sub=True)),             # ... and four rows a thread
    (5003, 10, "mse", dict(min_weight=40.0)),          # most leaves above the last level
    (4001, 10, "gaussian_mle", dict(weights=True, min_weight=9.0)),  # nodes of the last two levels that no level reached
])
def test_gradients_behind_the_tree(evt, N, D, loss, more):
    """With "grads_ahead" a small tree's last kernel adds the leaf values and computes the next gradients: the bits that the kernels of larger inputs
    and strictly alternating calls leave, also after a tree that keeps the predictions."""
    F, B, K = 5, 32, 3
    rng = np.random.default_rng(N + D)
    if loss == "mlogloss":
        x_bin = rng.integers(1, B + 1, size=(F, N), dtype=np.uint8)
        y, mu, w = (1 + (x_bin[0].astype(int) + rng.integers(0, 2, N)) % K).astype(np.float32), np.zeros(K, np.float32), None
    else:
        x_bin, y, w, mu = make_data(N, N, F, B, loss, more.get("weights", False))
    js = np.arange(1, F + 1, dtype=np.uint32)
    args = dict(eta=0.4, min_weight=more.get("min_weight", 0.0 if N < 10 else 2.0), L2=1.0)
    masks = [rng.integers(0, 256, N, dtype=np.uint8) for _ in range(5)]
    out = []
    for small, ahead in ((2, 1), (3, 1), (2, 0), (3, 0), (0, 1)):  # 2 is not taken above 65 535 rows
        h = evt.Handle(N, F, B, len(mu), D, loss, "oblivious" if more.get("oblivious") else "binary")
        h.set_option("small_tree", small)
        h.set_option("grads_ahead", ahead)
        h.set_xbin(x_bin)
        h.set_target(y, w, mu)
        rec = []
        for r in range(5):
            h.update_grads()
            gp = evt.make_params(update_pred=r != 3, **args)
            rec.append(h.grow_tree(js, gp, mask=masks[r] if more.get("sub") else None, cond=150))
            rec.append(h.get_hist())
            if r % 2:
                rec.append(h.get_pred())
        h.update_grads()
        rec += [h.get_grads(), np.concatenate(h.get_quant()), h.get_pred()]
        h.close()
        out.append(rec)
    for a in out[1:]:
        for one, other in zip(out[0], a):
            if isinstance(one, np.ndarray):
                assert one.tobytes() == other.tobytes()
            else:
                assert_tree_bits(one, other)
    assert sum(int(t.split.sum()) for t in out[0] if not isinstance(t, np.ndarray)) > 0 or N < 10
