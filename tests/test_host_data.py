"""Features in host memory on their way in: binning by the host's cores and the quantile edges, for every layout and type a program
may hold them in, against numpy's search in the order of isless and numpy's quantiles."""
import os
import subprocess
import threading

import numpy as np
import pytest


def _values(rng, kind, n):
    x = rng.standard_normal(n)
    if kind == "float32":
        x = x.astype(np.float32)
    elif kind == "tenths":  # Float64 values that are no Float32 and meet the edges
        x = np.round(x * 20) * 0.1
    elif kind == "whole":
        x = np.round(x * 5)
    elif kind == "huge":
        x = x * 1e300
    elif kind == "skewed":
        x = np.exp(9 * x)
    elif kind == "denormal":  # of the smallest value there is and zero
        x = np.where(x < 0, 0.0, 5e-324)
    elif kind == "tiny":  # a range whose reciprocal overflows
        x = x * 1e-310
    elif kind == "far":  # almost all values share one of any number of equal slices, and are tiny there
        x = np.where(rng.random(n) < 0.9, np.abs(x) * 1e-306, 1e-280)
    return x


def _search(e, v):
    """searchsortedfirst in the order of isless: NaN last, -0.0 before 0.0."""
    def key(a):
        a = np.asarray(a, np.float64)
        i = a.view(np.int64)
        k = np.where(i < 0, np.int64(-2 ** 63) - i - 1, i)
        return np.where(np.isnan(a), np.int64(2 ** 63 - 1), k)
    return (np.searchsorted(key(e), key(v), side="left") + 1).astype(np.uint8)


@pytest.mark.parametrize("kind", ["float32", "float64", "tenths", "whole", "huge"])
@pytest.mark.parametrize("shape", [(1, 1), (15, 3), (16, 16), (17, 17), (64, 33), (67, 5), (4200, 2)])
def test_bins_of_every_layout(evt, kind, shape):
    rng = np.random.default_rng(shape[0] + 7 * len(kind))
    N, F = shape
    edges = [np.sort(_values(rng, kind, rng.choice([1, 15, 16, 31, 63, 64, 127, 254])).astype(np.float64)) + 0.0 for _ in range(F)]
    x = _values(rng, kind, N * F).reshape(N, F)
    special = [np.nan, np.inf, -np.inf, 0.0, -0.0, 1e-310, edges[0][0], edges[-1][-1]]
    for v in special:
        x[rng.integers(N), rng.integers(F)] = v
    edges[0][np.abs(edges[0]) == 0] = -0.0  # compared value by value
    want = np.stack([_search(edges[j], x[:, j]) for j in range(F)])
    for lay, bins in ((x, want), (np.asfortranarray(x), want), (np.repeat(x, 2, axis=1)[:, ::2], want), (x[::-1], want[:, ::-1])):
        assert np.array_equal(evt.binarize(lay, edges), bins)


@pytest.mark.parametrize("kind", ["float32", "float64", "whole", "huge", "skewed", "denormal", "tiny", "far"])
@pytest.mark.parametrize("shape,nbins", [((1, 3), 4), ((64, 9), 2), ((65, 8), 255), ((3000, 17), 64), ((9000, 2), 8)])
def test_edges_are_numpys_quantiles(evt, kind, shape, nbins):
    rng = np.random.default_rng(1)
    x = _values(rng, kind, shape[0] * shape[1]).reshape(shape)
    x[0, 0] = np.inf
    x[-1, -1] = np.nan
    q = np.arange(1, nbins) / nbins
    for lay in (x, np.asfortranarray(x), x[:, ::-1][:, ::-1]):
        r1, r2 = np.random.default_rng(7), np.random.default_rng(7)
        edges, _, _ = evt.get_edges(lay, nbins, r1)
        n = min(shape[0], 1000 * nbins)
        idx = np.sort(r2.choice(shape[0], n, replace=False)) if n < shape[0] else np.arange(n)
        for j in range(shape[1]):
            col = np.asarray(x[idx, j], np.float64)
            want = np.quantile(col, q) if nbins > 2 else np.array([col.min()])
            assert np.array_equal(edges[j], want, equal_nan=True)


def test_more_columns_than_edges_are_refused(evt):
    with pytest.raises(IndexError):
        evt.binarize(np.zeros((50, 4)), [np.arange(3.0)] * 3)


class OneCore:
    """The calling thread on one core: there a large matrix goes up as it lies and is binned by the device."""

    def __enter__(self):
        self._was = os.sched_getaffinity(0)
        os.sched_setaffinity(0, {min(self._was)})

    def __exit__(self, *_):
        os.sched_setaffinity(0, self._was)


class Threads:
    """The most threads the process had at a look every half millisecond."""

    def __enter__(self):
        self.most, self._stop = 0, threading.Event()
        self._t = threading.Thread(target=self._look)
        self._t.start()
        return self

    def _look(self):
        while not self._stop.wait(0.0005):
            self.most = max(self.most, len(os.listdir("/proc/self/task")))

    def __exit__(self, *_):
        self._stop.set()
        self._t.join()


def test_callers_at_once_share_the_workers(evt):
    """Any number of calls at a time: right results, and in all no more worker threads than cores."""
    rng = np.random.default_rng(0)
    x, e = rng.random((400_000, 6)), np.sort(rng.random(63))
    want = evt.binarize(x, [e] * 6)
    same = [False] * 8

    def work(k):
        same[k] = all(np.array_equal(evt.binarize(x, [e] * 6), want) for _ in range(6))
    with Threads() as seen:
        callers = [threading.Thread(target=work, args=(k,)) for k in range(8)]
        before = len(os.listdir("/proc/self/task"))
        for t in callers:
            t.start()
        for t in callers:
            t.join()
    assert all(same)
    assert seen.most <= before + 8 + os.cpu_count() - 1


THROWING = r"""
#include "host_bin.h"
#include <cstdio>
#include <new>
#include <thread>
#include <unistd.h>
int main() {
    for (int rep = 0; rep < 50; rep++) {
        const std::thread::id caller = std::this_thread::get_id();
        std::atomic<int> done{0}, on_worker{0};
        bool caught = false;
        try { // the caller's own tasks are slow: workers take most of the others, and throw
            hb_parallel(64, 3, [&](int) {
                usleep(500);
                if (std::this_thread::get_id() != caller) {
                    on_worker++;
                    throw std::bad_alloc();
                }
                done++;
            });
        } catch (const std::bad_alloc &) {
            caught = true;
        }
        if (caught != (on_worker > 0) || (!caught && done != 64)) return 1;
        if (rep == 49 && !caught) return 2;
        std::atomic<int> after{0};
        hb_parallel(64, 3, [&](int) { after++; });
        if (after != 64) return 3;
    }
    puts("ok");
}
"""


def test_an_exception_of_a_worker_is_the_callers(evt, tmp_path):
    """The worker threads as they are, in a program of their own: an exception there ended the process."""
    if os.cpu_count() < 2:
        pytest.skip("no worker beside the caller")
    csrc = os.path.join(os.path.dirname(evt.__file__), "csrc")
    (tmp_path / "main.cpp").write_text(THROWING)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-x", "c++", "-O0", "-std=c++17", "-I", csrc, str(tmp_path / "main.cpp"), os.path.join(csrc, "host_bin.cpp"),
                    os.path.join(csrc, "host_bin_avx512.cpp"), "-o", exe, "-pthread"], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert (run.returncode, run.stdout) == (0, "ok\n"), run.stderr


AFFINITY = r"""
#include "host_bin.h"
#include <cstdio>
#include <sched.h>
#include <unistd.h>
int main() { // workers of a caller with few cores, then of one with all: each runs where its caller may
    cpu_set_t all, few, got;
    sched_getaffinity(0, sizeof(all), &all);
    CPU_ZERO(&few);
    for (int c = 0, n = 0; c < CPU_SETSIZE && n < 2; c++)
        if (CPU_ISSET(c, &all)) CPU_SET(c, &few), n++;
    for (const cpu_set_t *mine : {&few, &all, &few}) {
        sched_setaffinity(0, sizeof(*mine), mine);
        std::atomic<int> bad{0};
        hb_parallel(64, 3, [&](int) {
            usleep(300);
            cpu_set_t here;
            sched_getaffinity(0, sizeof(here), &here);
            if (!CPU_EQUAL(&here, mine)) bad++;
        });
        if (bad) return 1;
    }
    puts("ok");
}
"""


def test_workers_run_on_their_callers_cores(evt, tmp_path):
    csrc = os.path.join(os.path.dirname(evt.__file__), "csrc")
    (tmp_path / "main.cpp").write_text(AFFINITY)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-x", "c++", "-O0", "-std=c++17", "-I", csrc, str(tmp_path / "main.cpp"), os.path.join(csrc, "host_bin.cpp"),
                    os.path.join(csrc, "host_bin_avx512.cpp"), "-o", exe, "-pthread"], check=True)
    run = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert (run.returncode, run.stdout) == (0, "ok\n"), run.stderr


QUOTA = r"""
#include "host_bin.cpp"
int main(int, char **a) {
    printf("%d %d\n", quota_cores(a[1], a[2], a[3]) >> 20 ? -1 : quota_cores(a[1], a[2], a[3]), hb_cores());
}
"""


def test_cores_are_counted_within_affinity_and_quota(evt, tmp_path):
    csrc = os.path.join(os.path.dirname(evt.__file__), "csrc")
    (tmp_path / "main.cpp").write_text(QUOTA)
    exe = str(tmp_path / "main")
    subprocess.run(["g++", "-x", "c++", "-O0", "-std=c++17", "-I", csrc, str(tmp_path / "main.cpp"), os.path.join(csrc, "host_bin_avx512.cpp"), "-o", exe,
                    "-pthread"], check=True)
    for cpu_max, quota, period, want in (("max 100000", None, None, -1), ("1600000 100000", None, None, 16), ("150000 100000", None, None, 2),
                                         (None, "-1", "100000", -1), (None, "50000", "100000", 1), (None, None, None, -1), ("", "200000", "100000", 2)):
        files = []
        for name, text in (("max", cpu_max), ("quota", quota), ("period", period)):
            files.append(str(tmp_path / name))
            if text is None and os.path.exists(files[-1]):
                os.remove(files[-1])
            elif text is not None:
                open(files[-1], "w").write(text + "\n")
        one = min(os.sched_getaffinity(0))
        got = subprocess.run([exe] + files, capture_output=True, text=True, preexec_fn=lambda: os.sched_setaffinity(0, {one})).stdout
        assert got == "%d 1\n" % want


def test_the_smallest_and_largest_calls(evt):
    """No rows, no columns, no edges, more edges than a bin's byte counts (it wraps): what numpy's search gives."""
    rng = np.random.default_rng(0)
    assert evt.binarize(np.zeros((0, 3)), [np.arange(3.0)] * 3).shape == (3, 0)
    assert evt.binarize(np.zeros((3, 0)), []).shape == (0, 3)
    assert evt.binarize_table({"a": np.zeros(0)}, ["a"], [np.arange(3.0)]).shape == (1, 0)
    assert np.array_equal(evt.binarize(np.arange(4)[:, None], [()]), np.ones((1, 4)))
    for n in (254, 255, 256, 700):
        e, x = np.sort(rng.random(n)), rng.random((77, 3))
        want = np.stack([(np.searchsorted(e, x[:, j]) + 1).astype(np.uint8) for j in range(3)])
        assert np.array_equal(evt.binarize(x, [e] * 3), want) and np.array_equal(evt.binarize(np.asfortranarray(x), [e] * 3), want)
    for bad in (2.0, np.zeros((2, 2))):
        with pytest.raises(ValueError):
            evt.binarize(np.zeros((4, 1)), [bad])
    with pytest.raises(ValueError):
        evt.binarize(np.zeros((4, 2, 2)), [np.arange(3.0)] * 2)
    assert evt.get_edges(np.zeros((3, 0)), 16, rng)[0] == []
    assert [len(e) for e in evt.get_edges(np.zeros((3, 2)), 1, rng)[0]] == [0, 0]
    for nbins in (2, 16):
        with pytest.raises(IndexError):
            evt.get_edges(np.zeros((0, 3)), nbins, rng)


@pytest.mark.gpu
def test_a_handle_takes_one_feature_for_each_of_its_columns(evt):
    h = evt.Handle(50, 4, 16, 1, 3, "mse")
    for n in (3, 5):
        with pytest.raises(ValueError):
            h.binarize_matrix(np.zeros((50, 4)), [np.arange(3.0)] * n)
    h.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("order", ["C", "F"])
@pytest.mark.parametrize("shape", [(1, 40), (1000, 1), (77, 19), (70_001, 24), (400_003, 50), (9_000_001, 2)])
def test_upload_of_a_matrix_as_it_lies(evt, dtype, order, shape):
    """One piece, several, more pieces than buffers; rows and columns contiguous: the handle holds the host's bins."""
    rng = np.random.default_rng(3)
    N, F = shape
    x = np.asarray(rng.random(shape, np.float32) if N * F > 10 ** 6 else rng.random(shape), dtype, order=order)
    edges = [np.sort(rng.random(15)) for _ in range(F)]
    h = evt.Handle(N, F, 16, 1, 3, "mse")
    h.binarize_matrix(x, edges)
    assert np.array_equal(h.get_xbin(), evt.binarize(x, edges))
    h.close()


@pytest.mark.gpu
def test_leaf_ids_of_more_pieces_than_buffers(evt):
    """The ids of a piece are spread out while later pieces are binned, by the same workers."""
    from test_gpu_kept_model import _model
    rng = np.random.default_rng(6)
    m = _model(evt, rng, 4, 16, 1, "mse", [9] * 200)  # 2-byte ids, 404 bytes a row: ten pieces of 20k rows
    x = rng.random((200_000, 4), np.float32)
    want = evt._lib.predict_leaf_idx(evt.binarize(x, m.info["edges"]), m.info["feattypes"], m.trees)
    evt.predict_leaf_idx(m, x)
    before = len(os.listdir("/proc/self/task"))
    with Threads() as seen:
        got = evt.predict_leaf_idx(m, x)
    assert np.array_equal(got, want)
    assert seen.most <= before + 1


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("order", ["C", "F", "wide C", "wide F"])
@pytest.mark.parametrize("shape", [(70_001, 24), (1_000_003, 2), (400_003, 50), (17, 40_000), (300, 1030), (9_000_001, 2)])
def test_a_matrix_binned_by_the_device(evt, dtype, order, shape):
    """One piece, several, more than buffers; rows and columns contiguous, with gaps between them; edges that only isless tells apart."""
    rng = np.random.default_rng(3)
    N, F = shape
    x = np.asarray(rng.random((N + 3, F + 5), np.float32), dtype, order=order[-1])
    x = x[:N, :F] if "wide" in order else np.asarray(x[:N, :F], order=order)
    edges = [np.sort(np.float32(rng.random(rng.choice([1, 7, 15])))).astype(np.float64) for _ in range(F)]
    edges[0] = np.array([-0.0, 0.5, np.nan])
    edges[1] = np.sort(rng.random(254))
    for v in (np.nan, np.inf, -np.inf, 0.0, -0.0, 0.5):
        for j in (0, F - 1):
            x[rng.integers(N), j] = v
    h = evt.Handle(N, F, 255, 1, 3, "mse")
    with OneCore():
        h.binarize_matrix(x, edges)
    assert np.array_equal(h.get_xbin(), evt.binarize(x, edges))
    h.close()


@pytest.mark.gpu
@pytest.mark.parametrize("N,F,K,loss,depths", [(70_001, 24, 1, "mse", [6] * 9), (400_003, 5, 3, "mlogloss", [5] * 6), (40_000, 100, 2, "gaussian_mle", [4] * 300)])
def test_predictions_binned_by_the_device(evt, N, F, K, loss, depths):
    from test_gpu_kept_model import _check, _model
    rng = np.random.default_rng(N)
    m = _model(evt, rng, F, 64, K, loss, depths)
    x = rng.random((N, F), np.float32)
    want, leaf = evt.predict(m, x), evt.predict_leaf_idx(m, x)
    with OneCore():
        for lay in (x, np.asfortranarray(x), x.astype(np.float64), np.repeat(x, 2, axis=1)[:, ::2]):
            assert np.array_equal(evt.predict(m, lay), want) and np.array_equal(evt.predict_leaf_idx(m, lay), leaf)
        _check(evt, m, x)  # the whole-model calls too


@pytest.mark.gpu
@pytest.mark.parametrize("N", [(64 << 20) - 1, 64 << 20, (64 << 20) + 1, (72 << 20) - 1, (72 << 20) + (1 << 19) + 1])
def test_bins_of_more_than_a_buffer(evt, N):
    """Around the size from which pinned pieces are taken, whole pieces, a piece and a task more, a byte more and less."""
    x = np.random.default_rng(0).integers(1, 17, (1, N), dtype=np.uint8)
    h = evt.Handle(N, 1, 16, 1, 1, "mse")
    h.set_xbin(x)
    assert np.array_equal(h.get_xbin(), x)
    h.close()
