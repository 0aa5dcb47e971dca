"""Trees on every row whose rows are walked through them at the end give the predictions, gradients, node ids and following trees of those whose
rows leave their leaf's number, and of those whose leaf values are added while the last level is partitioned, bit for bit."""
import numpy as np
import pytest

from test_gpu_parity import assert_tree_bits, make_data

pytestmark = pytest.mark.gpu


LOSSES = [("mse", False), ("mse", True), ("logloss", False), ("poisson", True), ("gamma", False), ("tweedie", False), ("mae", False), ("gaussian_mle", False),
          ("logistic_mle", True)]


@pytest.mark.parametrize("loss,weights,N,F,D,tt", [(*lw, *s) for lw in LOSSES for s in ((63, 5, 3, "binary"), (8_001, 20, 6, "oblivious"))] +
                         [(*lw, *s) for lw in LOSSES if not lw[1] for s in ((600_007, 17, 5, "binary"), (2_100_001, 9, 4, "binary"))])
def test_walk_equals_words(evt, loss, weights, N, F, D, tt):
    x_bin, y, w, mu = make_data(N, N, F, 32, loss, weights)
    js = np.arange(1, F + 1, dtype=np.uint32)
    gp = evt.make_params(eta=0.3)
    out = []
    for defer in (2, 3, 0):
        h = evt.Handle(N, F, 32, mu.shape[0], D, loss, tt)
        h.set_option("small_tree", 0)
        h.set_option("grads_ahead", 1)
        h.set_option("defer_pred", defer)
        h.set_xbin(x_bin)
        h.set_target(y, w, mu)
        rec = []
        for _ in range(3):
            h.update_grads()
            t = h.grow_tree(js, gp)
            rec.append((t, h.get_pred(), h.get_grads(), h.get_nidx()))
        h.close()
        out.append(rec)
    for other in out[1:]:
        for a, b in zip(out[0], other):
            assert_tree_bits(a[0], b[0])
            for u, v in zip(a[1:], b[1:]):
                assert u.tobytes() == v.tobytes()
    assert N < 100 or out[0][0][0].split.any()


@pytest.mark.parametrize("loss,N", [("mse", 600_007), ("poisson", 2_100_001)])
def test_walk_of_weighted_rows_in_wide_blocks(evt, loss, N):
    """Blocks of 1024 threads of two and of four rows each, with weights."""
    test_walk_equals_words(evt, loss, True, N, 9, 4, "binary")


@pytest.mark.parametrize("loss,weights,tt", [("mse", False, "binary"), ("logloss", True, "binary"), ("gaussian_mle", False, "oblivious")])
def test_modes_follow_each_other_on_one_handle(evt, loss, weights, tt):
    """A tree that is walked behind one whose leaf values are still to be added, and the other way round, with samples of the columns; and small trees between them."""
    N, F, D = 30_011, 12, 5
    x_bin, y, w, mu = make_data(77, N, F, 32, loss, weights)
    gp = evt.make_params(eta=0.3)
    out = []
    for modes in ((3, 2, 3, 2, 2, 1, 3, 1, 2), (0,) * 9, (2,) * 9):
        h = evt.Handle(N, F, 32, mu.shape[0], D, loss, tt)
        h.set_option("grads_ahead", 1)
        h.set_xbin(x_bin)
        h.set_target(y, w, mu)
        rng = np.random.default_rng(5)
        rec = []
        for k, mode in enumerate(modes):
            h.set_option("small_tree", 2 if k == 4 and modes[0] == 3 else 0)
            h.set_option("defer_pred", mode)
            js = (np.sort(rng.choice(F, 7, replace=False)) + 1).astype(np.uint32)
            h.update_grads()
            rec.append((h.grow_tree(js, gp), h.get_pred() if k % 3 == 2 else None, h.get_nidx() if k % 4 == 1 else None))
        rec.append((None, h.get_pred(), h.get_grads()))
        h.close()
        out.append(rec)
    for other in out[1:]:
        for a, b in zip(out[0], other):
            if a[0] is not None:
                assert a[0].split.any()
                assert_tree_bits(a[0], b[0])
            for u, v in zip(a[1:], b[1:]):
                assert (u is None) == (v is None) and (u is None or u.tobytes() == v.tobytes())


def test_any_integer_means_on_or_off(evt):
    N, F = 4_001, 6
    x_bin, y, w, mu = make_data(N, N, F, 32, "mse", False)
    h = evt.Handle(N, F, 32, 1, 4, "mse")
    h.set_option("small_tree", 0)
    h.set_xbin(x_bin)
    first = None
    for value in (1, 4, 255, -1, -(1 << 40), 1 << 40, 0):
        h.set_option("defer_pred", value)
        h.set_target(y, w, mu)
        h.update_grads()
        got = (h.grow_tree(np.arange(1, F + 1, dtype=np.uint32), evt.make_params(eta=0.3)), h.get_pred())
        first = first or got
        assert_tree_bits(got[0], first[0])
        assert got[1].tobytes() == first[1].tobytes()
    h.close()
