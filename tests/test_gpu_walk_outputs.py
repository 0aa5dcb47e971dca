"""Kept models of more than two outputs, whose trees are added by a lane per row and output: each stride of the leaf values with and without
lanes past the last output, each clamp, on both sides of every change of the rows a block takes (values and leaf ids), bit for bit against
the calls that pack their trees every time."""
import numpy as np
import pytest

from test_gpu_kept_model import _check, _model

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K,loss", [(3, "mlogloss"), (4, "mlogloss"), (7, "mlogloss"), (8, "mlogloss"), (9, "mlogloss"), (16, "mlogloss"),
                                    (3, "mse"), (5, "logloss"), (6, "gaussian_mle"), (12, "logistic_mle")])
def test_outputs_and_rows_of_a_block(evt, K, loss):
    rng = np.random.default_rng(K)
    m = _model(evt, rng, 6, 32, K, loss, [1, 4, 6, 2, 5] * 5, True)  # 25 trees: whole runs of the trees read ahead, and a rest
    for t in m.trees:
        t.pred *= 8  # reaches the clamps
    if loss == "mlogloss":  # a class out of reach, and one alone in it
        m.trees[1].pred[::3, K - 1] = -np.inf
        m.trees[2].pred[::5, 0] = np.inf
    x = rng.random((32_769, 6), np.float32)
    for n in (1, 4, 5, 192, 193, 1024, 1025, 3072, 3073, 8192, 8193, 32_768, 32_769):
        _check(evt, m, x[:n])
