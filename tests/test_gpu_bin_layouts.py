"""The layouts made of the bins - records of rows, threshold planes - at the edges of the tiles they are made in: every row's bins are counted where they belong, trees
decided by planes are those decided by bins, and a bin out of range is found wherever it lies."""
import numpy as np
import pytest

from test_gpu_parity import assert_tree_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,F,B", [
    (3, 1, 2), (31, 16, 16), (33, 17, 17), (255, 5, 64), (256, 20, 33), (257, 31, 65), (1027, 100, 64), (4099, 129, 32), (2055, 260, 16), (8191, 7, 255), (70_001, 33, 128),
])
def test_records_and_planes(evt, N, F, B):
    rng = np.random.default_rng(N + F)
    x = rng.integers(1, B + 1, size=(F, N), dtype=np.uint8)
    y = (x[0] / B + x[F - 1] / B + 0.3 * rng.standard_normal(N)).astype(np.float32)
    js = np.arange(1, F + 1, dtype=np.uint32)
    gp = evt.make_params(eta=0.3, L2=1.0, min_weight=0.0)
    out = []
    for planes in (1, 0):
        h = evt.Handle(N, F, B, 1, 5, "mse")
        h.set_option("small_tree", 0)
        h.set_option("bit_planes", planes)
        h.set_xbin(x)
        h.set_target(y, None, np.zeros(1, np.float32))
        rec = []
        for r in range(3):
            h.update_grads()
            rec.append(h.grow_tree(js, gp))
            if r == 0:  # the root's row counts, exactly
                hist = h.get_hist()
                counts = np.asarray(hist).reshape(-1, F, B, 3)[0, :, :, 2]
                want = np.stack([np.bincount(x[j].astype(int) - 1, minlength=B) for j in range(F)])
                assert np.array_equal(counts, want)
            rec.append(h.get_nidx())
        rec.append(h.get_pred())
        out.append(rec)
        h.close()
    for a, b in zip(*out):
        if isinstance(a, np.ndarray):
            assert a.tobytes() == b.tobytes()
        else:
            assert_tree_bits(a, b)


@pytest.mark.parametrize("row", [0, 255, 256, 1027])
@pytest.mark.parametrize("feat", [0, 16, 99])
def test_a_bin_out_of_range_is_found(evt, row, feat):
    N, F, B = 1028, 100, 64
    x = np.ones((F, N), np.uint8)
    h = evt.Handle(N, F, B, 1, 4, "mse")
    h.set_xbin(x)
    for bad in (0, B + 1, 255):
        x[feat, row] = bad
        with pytest.raises(evt.EvtError):
            h.set_xbin(x)
    x[feat, row] = B
    h.set_xbin(x)
    h.close()
