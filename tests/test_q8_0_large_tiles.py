"""The batched Q8_0 GEMM over large tiles (frk_gemm_q8_pipe.hip) at the edges of its tiles, stages and splits."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import fa, to_dev  # noqa: F401 (fa: the module's fixture)


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,batch", [
    (14337, 1024, 513),   # 256 x 128 tiles, a row and a token past the last whole ones
    (8192, 1056, 1000),   # 33 blocks: the last half chunk holds one, the next none
    (11008, 352, 200),    # 128 x 64 tiles, a last half chunk of three blocks
    (1024, 2080, 130),    # few tiles: the columns split four ways, the last part the shortest
    (130, 8192, 65), (3000, 32, 700),
])
def test_large_tiles_match_exact_arithmetic(fa, rows, cols, batch):
    from bench import random_blocks
    from frink_amd import synth
    print("q8_0 large tiles", rows, cols, batch, flush=True)
    data = random_blocks(fo.Q8_0, rows, cols, seed=rows)
    x = synth.activations(batch, batch, cols, outlier_frac=0.01)
    w = fa.Weights.from_host(fo.Q8_0, data, rows, cols)
    got = w.gemm(to_dev(x)).cpu().numpy().astype(np.float64)
    w.release()
    xb = x.reshape(batch, cols // 32, 32)
    amax = np.abs(xb).max(axis=2)
    inv = np.where(amax != 0, np.float32(127) / np.where(amax != 0, amax, 1), 0).astype(np.float32)
    q = np.clip(np.rint(xb * inv[:, :, None]), -127, 127).astype(np.float64)
    a = (q * (amax / np.float32(127)).astype(np.float16).astype(np.float64)[:, :, None]).reshape(batch, cols)
    wd = fo.dequant(fo.Q8_0, data).reshape(rows, cols).astype(np.float64)
    # a block's term is exact up to its addition: one f32 rounding a block, and one a part of a split (four at most)
    room = (cols // 32 + 4) * 2.0 ** -24 * (np.abs(a) @ np.abs(wd).T)
    assert (np.abs(got - a @ wd.T) <= room).all()


def test_no_result_of_the_matrix_core_is_read_too_soon(tmp_path):
    import isa_mfma_lint
    from test_isa_waits import _assembly
    asm = _assembly(tmp_path, "frk_gemm_q8_pipe.hip")
    assert "v_mfma_i32_32x32x32_i8" in asm
    assert isa_mfma_lint.violations(asm) == []
