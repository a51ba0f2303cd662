"""A row of Q4_K and Q5_K on the kernel whose wavefronts take whole rows, in the one-launch form that quantizes inside (from 17 blocks, where
the rows fill the chip with three a wavefront or, Q5_K, two): row counts that fill a workgroup's spans and fall short of one."""
import pytest

import oracle as fo
from test_gpu_parity import assert_rows_close, fa, to_dev  # noqa: F401 (fa: the module's fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,rows,blocks", [(fo.Q4_K, 4097, 17), (fo.Q4_K, 6144, 20), (fo.Q4_K, 4321, 19), (fo.Q4_K, 8209, 18), (fo.Q5_K, 4097, 17), (fo.Q5_K, 6143, 20),
                                              (fo.Q5_K, 2049, 21), (fo.Q5_K, 4100, 31), (fo.Q5_K, 8210, 21)])
def test_whole_rows_in_one_launch(fa, kind, rows, blocks):
    from bench import random_blocks
    from frink_amd import synth
    print("whole rows", kind, rows, blocks, flush=True)
    cols = 256 * blocks
    data = random_blocks(kind, rows, cols, rows + cols)
    x = synth.activations(rows + cols, 1, cols, outlier_frac=0.01)[0]
    w = fa.Weights.from_host(kind, data, rows, cols)
    assert_rows_close(w.gemv(to_dev(x)).cpu().numpy()[None], fo.gemv(kind, data, rows, cols, x, fo.INT_DOT)[None], "whole rows %dx%d" % (rows, cols))
    w.release()
