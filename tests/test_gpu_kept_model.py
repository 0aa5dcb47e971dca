"""Predictions of a kept model (evt_model_predict) against the whole-model calls that pack their trees every time, bit for bit: every
rows-per-block of the row kernel and the hand-over to the 1024-row kernel, output counts, tree sizes, feature counts."""
import numpy as np
import pytest

from test_gpu_lifecycle import _free_bytes
from test_gpu_parity import _random_tree

pytestmark = pytest.mark.gpu


def _model(evt, rng, F, B, K, loss, depths, cat=False):
    trees = []
    for d in depths:
        r, t = _random_tree(rng, d, F, B, K), evt.Tree(K, (1 << d) - 1)
        for f in ("feat", "cond_bin", "pred", "split"):
            getattr(t, f)[...] = getattr(r, f)
        trees.append(t)
    ft = (rng.random(F) > 0.3).astype(np.uint8) if cat else np.ones(F, np.uint8)
    return evt.EvoTree(loss, K, trees, dict(edges=[np.sort(rng.random(B - 1)) for _ in range(F)], feattypes=ft, feature_names=["f%d" % j for j in range(F)]))


def _check(evt, m, x, n=None):
    L = evt._lib
    trees, ft = m.trees[:n], m.info["feattypes"]
    want = L.predict_model_f64(np.ascontiguousarray(x.T, np.float64), m.info["edges"], ft, m.loss_type, m.K, trees)
    got = evt.predict(m, x, ntree_limit=n)
    assert np.array_equal(got.reshape(want.shape).view(np.uint32), want.view(np.uint32))
    assert np.array_equal(evt.predict_leaf_idx(m, x, ntree_limit=n), L.predict_leaf_idx(evt.binarize(x, m.info["edges"]), ft, trees))


@pytest.mark.parametrize("N,F,B,K,loss,depths,cat", [
    (1, 1, 2, 1, "mse", [1], False),
    (1, 20, 64, 1, "mse", [1] + [6] * 100, False),
    (3, 7, 16, 2, "gaussian_mle", [1, 4, 2, 5, 7], True),
    (1024, 28, 128, 1, "logloss", [1] + [8] * 40, False),
    (1025, 5, 32, 4, "mlogloss", [6, 3, 6], True),
    (8193, 13, 255, 16, "mlogloss", [5] * 70, False),
    (65_537, 3, 8, 5, "mlogloss", [9, 1, 9], False),
    (140_001, 9, 32, 1, "mse", [6] * 9, True),
    (300_001, 30, 32, 2, "gaussian_mle", [1] + [6] * 5, False),
    (130, 1030, 16, 1, "mse", [9] * 6, False),
    (5, 40_000, 4, 1, "mse", [10] * 3, False),
    (70, 4, 16, 1, "mse", [3] * 2100, False),
])
def test_equals_the_unkept_calls(evt, N, F, B, K, loss, depths, cat):
    rng = np.random.default_rng(N + F)
    m = _model(evt, rng, F, B, K, loss, depths, cat)
    x = rng.random((N, F), np.float32)
    _check(evt, m, x)
    _check(evt, m, np.asfortranarray(x.astype(np.float64)), max(1, len(depths) // 2))


def test_follows_changes_of_the_model(evt):
    rng = np.random.default_rng(9)
    m = _model(evt, rng, 6, 32, 1, "mse", [5] * 8)
    x = rng.random((50, 6))
    _check(evt, m, x)
    m.trees[3].pred *= 2  # in place
    _check(evt, m, x)
    m.trees[2].pred = m.trees[2].pred + 1  # another array
    _check(evt, m, x)
    m.info["edges"][1] += 0.01
    _check(evt, m, x)
    m.info["edges"][2] = m.info["edges"][2][:7] * 0.5
    _check(evt, m, x)
    m.trees[4] = m.trees[0]
    m.trees.append(m.trees[1])
    _check(evt, m, x)
    with pytest.raises(ValueError):
        evt.predict(m, np.zeros((3, 7)))
    m.trees[1].split[-1] = 1  # a split node whose children do not exist
    m.trees[1].feat[-1] = 1
    with pytest.raises(evt.EvtError):
        evt.predict(m, x)


def test_takes_what_the_whole_model_calls_take(evt):
    rng = np.random.default_rng(4)
    # leaf ids of so many trees that 64 rows of them do not fit a piece's buffer
    m = _model(evt, rng, 3, 16, 1, "mse", [9] * 3)
    m.trees = m.trees * 22_000
    x = rng.random((3, 3))
    assert np.array_equal(evt.predict_leaf_idx(m, x), np.tile(evt.predict_leaf_idx(m, x, ntree_limit=3), (1, 22_000)))
    # trees behind the limit that the matrix is too narrow for, or that are none
    m = _model(evt, rng, 3, 16, 1, "mse", [5] * 4)
    wide = _model(evt, rng, 6, 16, 1, "mse", [5] * 4)
    m.trees += wide.trees
    x = rng.random((70, 3))
    want = evt._lib.predict_model_f64(np.ascontiguousarray(x.T), m.info["edges"], m.info["feattypes"], "mse", 1, m.trees[:4])
    assert np.array_equal(evt.predict(m, x, ntree_limit=4), want.reshape(-1))
    with pytest.raises(evt.EvtError):
        evt.predict(m, x)
    m.trees[7].split[-1] = m.trees[7].feat[-1] = 1
    assert np.array_equal(evt.predict(m, x, ntree_limit=4), want.reshape(-1))
    for n in (2, 4):  # neither fewer columns than features nor more
        with pytest.raises(ValueError):
            evt.predict(m, rng.random((5, n)), ntree_limit=4)


def test_what_models_keep_is_bounded_and_given_back(evt):
    """Twelve models that would keep 860 MB on the device and 1.8 GB beside it: 1 GB at most stays, and nothing after a trim."""
    rng = np.random.default_rng(5)
    x = rng.random((3, 4), np.float32)
    models = []
    for _ in range(12):
        m = _model(evt, rng, 4, 16, 16, "mse", [11])
        m.trees = m.trees * 1000
        models.append(m)
    evt.predict(models[0], x)
    evt._lib.trim()
    free = _free_bytes()
    want = [evt.predict(m, x) for m in models]
    assert 0 < free - _free_bytes() < 500 << 20
    for m, w in zip(models, want):  # those that went are packed again
        assert np.array_equal(evt.predict(m, x), w)
    evt._lib.trim()
    assert _free_bytes() >= free
    for m, w in zip(models[:2], want):
        assert np.array_equal(evt.predict(m, x), w)


def test_calls_of_several_threads_on_several_models(evt):
    import threading
    rng = np.random.default_rng(8)
    x = rng.random((700, 6))
    models = [_model(evt, rng, 6, 32, 1, "mse", [5] * 8) for _ in range(3)]
    want = [evt.predict(m, x) for m in models]
    same = [False] * 6

    def work(k):
        same[k] = all(np.array_equal(evt.predict(models[(k + i) % 3], x), want[(k + i) % 3]) for i in range(40))
    threads = [threading.Thread(target=work, args=(k,)) for k in range(6)]
    for t in threads:
        t.start()
    for _ in range(10):
        evt._lib.trim()  # beside them
    for t in threads:
        t.join()
    assert all(same)


def test_replaced_arrays_are_noticed_whatever_other_trees_do(evt):
    """Replacements beside each other on many threads, on this model's trees and on others'; copies of a model; trees of a fit."""
    import copy
    import pickle
    import threading
    rng = np.random.default_rng(10)
    x, y = rng.random((300, 5)), rng.random(300)
    m = evt.fit(evt.EvoTreeRegressor(nrounds=6, max_depth=4), x_train=x, y_train=y, verbosity=0)
    _check(evt, m, x)
    for c in (copy.deepcopy(m), pickle.loads(pickle.dumps(m))):
        _check(evt, c, x)
        c.trees[3].pred = c.trees[3].pred * 2
        _check(evt, c, x)
    _check(evt, m, x)
    # an assignment to another model's tree leaves this one's addresses as they are
    kept = evt._kept[m]
    before = kept._tree
    evt.Tree(1, 3).pred = np.zeros((3, 1), np.float32)
    c.trees[0].pred = c.trees[0].pred + 1
    evt.predict(m, x)
    assert kept._tree is before
    stop = threading.Event()

    def replace(k):
        while not stop.is_set():
            m.trees[1 + k].pred = m.trees[1 + k].pred * np.float32(1)
    threads = [threading.Thread(target=replace, args=(k,)) for k in range(4)]
    for t in threads:
        t.start()
    for _ in range(40):
        m.trees[6].pred = m.trees[6].pred + np.float32(0.5)
        _check(evt, m, x[:20])
    stop.set()
    for t in threads:
        t.join()
