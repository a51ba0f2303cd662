"""Q8_0 batches of up to 64 rows (gemm_q8_0_rows_kernel, frk_gemm_q8_pipe.hip) at the edges of its rows, lines of tokens, half
chunks of 128 columns and splits, against 64-bit sums of the same quants."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import fa, to_dev  # noqa: F401 (fa: a fixture)


@pytest.mark.gpu
@pytest.mark.parametrize("batch,rows,cols", [
    (2, 1, 32), (3, 31, 96), (8, 33, 128), (9, 32, 160), (16, 65, 1056), (17, 64, 992), (32, 97, 1024), (31, 1, 2144),
    (33, 65, 1056), (40, 33, 2080), (64, 97, 992), (48, 32, 96),
    (5, 33, 14336), (44, 100, 8224), (12, 100, 8224), (32, 2048, 3104),  # rows split between workgroups; many of them
])
def test_small_batches(fa, batch, rows, cols):
    rng = np.random.default_rng(batch + rows + cols)
    blk = np.zeros((rows, cols // 32, 34), np.uint8)
    dw = (rng.uniform(2e-4, 2e-2, (rows, cols // 32)) * rng.choice([-1.0, 1.0], (rows, cols // 32))).astype(np.float16)
    qw = rng.integers(-128, 128, (rows, cols // 32, 32)).astype(np.int8)
    blk[:, :, :2], blk[:, :, 2:] = dw.view(np.uint8).reshape(rows, -1, 2), qw.view(np.uint8)
    x = rng.standard_normal((batch, cols)).astype(np.float32)
    x[0, :32] = 0
    w = fa.Weights.from_host(fo.Q8_0, blk.reshape(-1), rows, cols)
    xd = to_dev(x)
    got, again = w.gemm(xd).cpu().numpy(), w.gemm(xd).cpu().numpy()
    w.release()
    xb = x.reshape(batch, cols // 32, 32)
    amax = np.abs(xb).max(axis=2)
    inv = np.where(amax != 0, np.float32(127) / np.where(amax != 0, amax, 1), 0).astype(np.float32)
    q = np.clip(np.rint(xb * inv[:, :, None]), -127, 127).astype(np.float64)
    a = (q * (amax / np.float32(127)).astype(np.float16).astype(np.float64)[:, :, None]).reshape(batch, cols)
    wd = (qw.astype(np.float64) * dw.astype(np.float64)[:, :, None]).reshape(rows, cols)
    # one rounding a block, then at most 8 wavefronts' sums of up to 8 workgroups
    room = (cols // 32 + 16) * 2.0 ** -24 * (np.abs(a) @ np.abs(wd).T)
    assert (np.abs(got - a @ wd.T) <= room).all()
    assert np.array_equal(got, again)
