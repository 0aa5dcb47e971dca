"""Trees of one launch (option "small_tree" = 4): every form of the kernel and every loss whose next gradients it computes, at sizes that it does take - which a
profiled tree shows: one launch, and none of the histogram and search kernels - against those kernels (= 0), bit for bit."""
import numpy as np
import pytest

from test_gpu_parity import assert_tree_bits, make_data, n_outputs

pytestmark = pytest.mark.gpu

LDS = 148 * 1024  # of a block


def hist_and_row_bytes(loss, F, B, weights):
    """LDS of the histograms of two levels, and of a row: its record, words, predictions, target, weight and place in two lists."""
    K = n_outputs(loss)
    rows = 4 if K == 2 else 1 if loss in ("mse", "mae") else 2  # gradient rows that are summed
    na = rows + (1 if weights else 0)
    return 16 * F * na * B, -(-F // 16) * 16 + 8 * na + (4 if weights else -4) + 4 * K + 4 + 4


def most_rows(loss, F, B, weights):
    hist, row = hist_and_row_bytes(loss, F, B, weights)
    return (LDS - hist) // row


def same(a, b):
    assert len(a) == len(b)
    for s, t in zip(a, b):
        if isinstance(s, np.ndarray):
            assert s.tobytes() == t.tobytes()
        else:
            assert_tree_bits(s, t)


def rounds(evt, form, N, F, B, D, loss, weights, ahead=1, sub=False, R=4):
    """What R free-running rounds leave, and the launches of the third by kernel class."""
    rng = np.random.default_rng(N + F)
    x_bin, y, w, mu = make_data(N + B, N, F, B, loss, weights)
    masks = [rng.integers(0, 256, N, dtype=np.uint8) for _ in range(R)]
    js = np.arange(1, F + 1, dtype=np.uint32)
    params = evt.make_params(eta=0.3, min_weight=0.0 if N < 10 else 2.0, L2=1.0)
    h = evt.Handle(N, F, B, len(mu), D, loss)
    try:
        h.set_option("grads_ahead", ahead)
        h.set_option("small_tree", form)
        h.set_xbin(x_bin)
        h.set_target(y, w, mu)
        rec, launches = [], {}
        for r in range(R):
            h.set_profiling(r == 2)
            h.update_grads()
            rec.append(h.grow_tree(js, params, mask=masks[r] if sub else None, cond=170))
            if r == 2:
                launches = {k: v["launches"] for k, v in h.get_profile().items()}
            rec += [h.get_hist(), h.get_nidx(), h.get_pred()]
        h.update_grads()
        return rec + [h.get_grads(), np.concatenate(h.get_quant())], launches
    finally:
        h.close()


def is_one_launch(launches):
    return launches["hist"] == 0 and launches["scan"] == 0 and launches["partition"] == 1


# Channels (2, 3, 5) x bins a lane (1, 2, 4) x weights; rows None: as many as it takes
@pytest.mark.parametrize("N,F,B,D,loss,weights,sub", [
    (None, 4, 33, 4, "mse", False, True),
    (2003, 64, 32, 5, "mse", True, False),
    (1031, 16, 128, 6, "mae", False, False),
    (1025, 17, 65, 5, "mae", True, True),
    (None, 5, 255, 7, "mse", False, False),
    (1201, 9, 129, 4, "mse", True, True),
    (None, 33, 16, 6, "logloss", False, True),
    (1501, 7, 64, 8, "poisson", True, False),
    (1999, 8, 100, 5, "gamma", False, False),
    (None, 5, 128, 6, "tweedie", True, True),
    (777, 6, 255, 4, "cred_var", False, True),
    (None, 3, 200, 9, "cred_std", True, False),
    (1601, 10, 64, 6, "gaussian_mle", False, False),
    (None, 9, 40, 5, "logistic_mle", True, True),
    (1023, 7, 96, 4, "logistic_mle", False, True),
    (None, 6, 100, 6, "gaussian_mle", True, False),
    (513, 5, 255, 3, "gaussian_mle", False, False),
    (None, 5, 200, 5, "logistic_mle", True, True),
])
def test_every_form_runs_and_changes_nothing(evt, N, F, B, D, loss, weights, sub):
    most = most_rows(loss, F, B, weights)
    N = most if N is None else min(N, most)
    others, launches = rounds(evt, 0, N, F, B, D, loss, weights, sub=sub)
    assert not is_one_launch(launches) and launches["hist"] > 0
    assert sum(int(t.split.sum()) for t in others if not isinstance(t, np.ndarray)) > 0
    for ahead in (0, 1):
        rec, launches = rounds(evt, 4, N, F, B, D, loss, weights, ahead, sub)
        assert is_one_launch(launches)
        same(rec, others)


@pytest.mark.parametrize("more_than,N,F,B,D,loss,weights", [
    ("rows in LDS", most_rows("mse", 4, 33, False), 4, 33, 5, "mse", False),
    ("rows in LDS", most_rows("mse", 1, 2, False), 1, 2, 2, "mse", False),  # the most of all
    ("rows in LDS", most_rows("gaussian_mle", 9, 64, True), 9, 64, 5, "gaussian_mle", True),
    ("features", 300, 64, 16, 4, "mse", False),
    ("depth", 900, 5, 16, 10, "mse", False),
])
def test_the_last_size_it_takes_and_the_next(evt, more_than, N, F, B, D, loss, weights):
    shapes = {"rows in LDS": (N + 1, F, D), "features": (N, F + 1, D), "depth": (N, F, D + 1)}
    for (n, f, d), takes in (((N, F, D), True), (shapes[more_than], False)):
        rec, launches = rounds(evt, 4, n, f, B, d, loss, weights)
        assert is_one_launch(launches) == takes
        same(rec, rounds(evt, 0, n, f, B, d, loss, weights)[0])


@pytest.mark.parametrize("N,takes", [(3, False), (4, True)])
def test_the_fewest_rows(evt, N, takes):
    rec, launches = rounds(evt, 4, N, 3, 8, 3, "mse", False)
    assert is_one_launch(launches) == takes
    same(rec, rounds(evt, 0, N, 3, 8, 3, "mse", False)[0])
