"""The evaluation metric in two halves: the value of the predictions as they stood at the first, whatever is queued in between."""
import numpy as np
import pytest

from test_gpu_parity import make_data

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,loss,metric", [(1, "mse", "rmse"), (1000, "logloss", "logloss"), (70_001, "gaussian_mle", "gaussian_mle")])
def test_metric_in_two_halves(evt, N, loss, metric):
    F, B, D = 4, 32, 4
    x_bin, y, w, mu = make_data(N, max(N, 600), F, B, loss, True)
    h = evt.Handle(x_bin.shape[1], F, B, len(mu), D, loss)
    h.set_xbin(x_bin)
    h.set_target(y, w, mu)
    h.update_grads()
    tree = h.grow_tree(np.arange(1, F + 1, dtype=np.uint32), evt.make_params(eta=0.3))
    e = evt.Handle(N, F, B, len(mu), 1, loss)
    e.set_xbin(np.ascontiguousarray(x_bin[:, :N]))
    e.set_target(y[:N], w[:N], mu)
    with pytest.raises(evt.EvtError):
        e.eval_metric_end()
    want = []
    for _ in range(3):
        e.predict_tree(tree)
        want.append(e.eval_metric(metric))
    e.set_target(y[:N], w[:N], mu)
    e.predict_tree(tree)
    for k in range(3):
        e.eval_metric_begin(metric)
        e.predict_tree(tree)  # behind it
        assert e.eval_metric_end() == want[k]
    with pytest.raises(evt.EvtError):
        e.eval_metric_end()
    tree.feat.setflags(write=False)  # arrays that give no writable buffer pass all the same
    tree.pred.setflags(write=False)
    e.predict_tree(tree)
    e.close()
    h.close()


@pytest.mark.parametrize("rounds", [1, 2, 3, 12])
def test_a_fit_that_queues_ahead_of_its_evaluation(evt, rounds):
    rng = np.random.default_rng(rounds)
    x, y = rng.random((900, 5)), rng.random(900)
    config = evt.EvoTreeRegressor(nrounds=rounds, max_depth=4, rowsample=0.7, early_stopping_rounds=2)
    args = dict(x_train=x[:600], y_train=y[:600], x_eval=x[600:], y_eval=y[600:], verbosity=0)
    a = evt.fit(config, **args)
    b, cache = evt.fit(config, return_cache=True, **args)  # keeps the handle: in turn
    cache.handle.close()
    assert a.info["logger"]["metrics"] == b.info["logger"]["metrics"] and len(a.trees) == len(b.trees)
    for s, t in zip(a.trees, b.trees):
        assert np.array_equal(s.feat, t.feat) and s.pred.tobytes() == t.pred.tobytes()


@pytest.mark.parametrize("patience", [1, 2, 5])
def test_early_stopping_drops_one_tree(evt, monkeypatch, patience):
    """Of the trees queued ahead of the evaluation that ends a fit, one at most is grown for nothing."""
    rng = np.random.default_rng(patience)
    x, y = rng.random((900, 5)), rng.random(900)  # noise: the metric soon stops improving
    queued, begin = [], evt._begin_tree
    monkeypatch.setattr(evt, "_begin_tree", lambda *args: (queued.append(1), begin(*args))[1])
    config = evt.EvoTreeRegressor(nrounds=60, max_depth=4, eta=0.3, early_stopping_rounds=patience)
    m = evt.fit(config, x_train=x[:600], y_train=y[:600], x_eval=x[600:], y_eval=y[600:], verbosity=0)
    kept = len(m.trees) - 1
    assert kept < 58 and len(queued) == kept + 1
