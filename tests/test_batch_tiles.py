"""The pipelined K-quant GEMM where its tiles are not filled.  Batches of 9 to 32 rows on the 64 x 32 tiles: rows past the last whole
tile, blocks that do not divide by a step's four shares, parts of few blocks, and the sizes on both sides of the rule that
sends a batch there.  Larger ones whose last token tile has few rows in use."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import fa, to_dev  # noqa: F401 (fa: the module's fixture)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", [
    (fo.Q4_K, 64, 256, 17), (fo.Q4_K, 65, 512, 32), (fo.Q4_K, 127, 1280, 31), (fo.Q4_K, 1000, 7680, 9), (fo.Q4_K, 4160, 2304, 20),
    (fo.Q4_K, 33, 14336, 16), (fo.Q5_K, 64, 2560, 17), (fo.Q5_K, 70, 8192, 9), (fo.Q5_K, 300, 2816, 32), (fo.Q5_K, 8200, 2304, 33),
    (fo.Q5_K, 4700, 6144, 10), (fo.Q6_K, 1300, 6912, 17), (fo.Q6_K, 2400, 11008, 13), (fo.Q6_K, 2700, 7936, 32), (fo.Q6_K, 4200, 4352, 25),
    (fo.Q6_K, 4161, 12288, 9), (fo.Q6_K, 700, 7936, 33),
])
def test_batches_match_exact_arithmetic(fa, kind, rows, cols, batch):
    _check(fa, kind, rows, cols, batch)


def _check(fa, kind, rows, cols, batch):
    from bench import random_blocks
    from frink_amd import synth
    print("batch tiles", kind, rows, cols, batch, flush=True)
    data = random_blocks(kind, rows, cols, seed=rows + cols)
    x = synth.activations(batch, batch, cols, outlier_frac=0.01)
    w = fa.Weights.from_host(kind, data, rows, cols)
    got = w.gemm(to_dev(x)).cpu().numpy().astype(np.float64)
    w.release()
    a = np.empty((batch, cols), np.float64)
    for r in range(batch):
        q, d, _ = fo.quantize_q8_k(x[r])
        a[r] = (q.reshape(-1, 256).astype(np.float64) * d.astype(np.float64)[:, None]).ravel()
    wd = fo.dequant(kind, data).reshape(rows, cols).astype(np.float64)
    # Integers are exact up to the float step: a handful of f32 roundings a block (sum, scale, mins) of terms no larger than
    # the block's sum of magnitudes, one for each addition onto the running sum, one a share and one a part.  The dequantized
    # weights round twice an element.  (Mins: the two terms of a block cancel, each is bounded by |a| times the offsets.)
    mag = np.abs(a) @ np.abs(wd).T
    if kind != fo.Q6_K:
        mag = mag + np.abs(a).sum(1)[:, None] * np.abs(wd).max(1)[None, :]
    room = (cols // 256 + 24) * 2.0 ** -24 * mag
    assert (np.abs(got - a @ wd.T) <= room).all(), float((np.abs(got - a @ wd.T) / room).max())


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", [
    (fo.Q4_K, 3000, 8192, 65), (fo.Q5_K, 2000, 8192, 97), (fo.Q6_K, 1024, 11008, 96), (fo.Q4_K, 2600, 8192, 129), (fo.Q5_K, 11008, 4096, 197),
    (fo.Q6_K, 11000, 4096, 170), (fo.Q4_K, 5000, 4352, 161), (fo.Q5_K, 8200, 2048, 225), (fo.Q6_K, 2900, 8192, 290), (fo.Q4_K, 3300, 6400, 321),
])
def test_last_token_tile_with_fewer_rows_in_use(fa, kind, rows, cols, batch):
    """One to three 32-token tiles of the last 128 in use, with and without parts of its own number."""
    _check(fa, kind, rows, cols, batch)
