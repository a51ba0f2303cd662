"""The host-buffer entry points' page-locked staging: results that end inside a chunk, at its edge and one past it, on both sides of
the size that goes through it, several outputs across chunks, several threads; the device entry points' bits."""
import threading

import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import bits, fa, make_weights, to_dev  # noqa: F401 (fa: the module's fixture)

pytestmark = pytest.mark.gpu


def _matrix(fa, rows, cols=256):
    base = make_weights(fo.Q4_K, min(rows, 509), cols, seed=rows).reshape(min(rows, 509), -1)
    data = np.ascontiguousarray(np.tile(base, ((rows + 508) // 509, 1))[:rows]).reshape(-1)
    return data, fa.Weights.from_host(fo.Q4_K, data, rows, cols)


@pytest.mark.parametrize("rows", [1, 3, 2047, 2048, 2049, 4097, 262143, 262144, 262145])  # (2048 floats a chunk, 262144 in all)
def test_one_result(fa, rows):
    print("host staging", rows, flush=True)
    data, w = _matrix(fa, rows)
    for seed in (1, 2):  # (the second finds the first one's results and flags in the staging memory)
        x = np.random.default_rng(seed).standard_normal(256).astype(np.float32)
        got = fa.launch_matvec(fo.Q4_K, data, x, rows, data.size // rows)
        assert np.array_equal(bits(got), bits(w.gemv(to_dev(x)).cpu().numpy()))
    w.release()


def test_several_results_and_a_batch(fa):
    sizes = [5, 2043, 2048, 1, 4100]
    pairs = [_matrix(fa, r) for r in sizes]
    x = np.random.default_rng(3).standard_normal(256).astype(np.float32)
    outs = fa.launch_matvec_multi(x, [fa.MatvecLaunch.of(fo.Q4_K, d, r, d.size // r) for (d, _), r in zip(pairs, sizes)])
    for got, (_, w) in zip(outs, pairs):
        assert np.array_equal(bits(got), bits(w.gemv(to_dev(x)).cpu().numpy()))
    data, w = pairs[4]
    xb = np.random.default_rng(4).standard_normal((70, 256)).astype(np.float32)
    for b in (1, 63, 64, 70):  # (4100 floats a row: 64 rows are past 1 MB)
        got = fa.launch_mul_mm(fo.Q4_K, data, xb[:b], 4100, 256, b, data.size // 4100)
        assert np.array_equal(bits(got), bits(w.gemm(to_dev(xb[:b])).cpu().numpy())), b
    for _, v in pairs:
        v.release()


def test_threads(fa):
    pairs = [_matrix(fa, r) for r in (700, 3000, 9000)]
    want, x = [], [np.random.default_rng(i).standard_normal(256).astype(np.float32) for i in range(3)]
    for (_, w), v in zip(pairs, x):
        want.append(bits(w.gemv(to_dev(v)).cpu().numpy()))
    wrong = []

    def work(i):
        data = pairs[i][0]
        rows = want[i].size
        for _ in range(40):
            if not np.array_equal(bits(fa.launch_matvec(fo.Q4_K, data, x[i], rows, data.size // rows)), want[i]):
                wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    for _, w in pairs:
        w.release()
