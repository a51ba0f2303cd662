"""The forms of the decode GEMV.  A row of Q4_K and Q5_K on the kernel whose wavefronts take whole rows, in the one-launch form that quantizes
inside (from 17 blocks, where the rows fill the chip with three a wavefront or, Q5_K, two): row counts that fill a workgroup's spans and
fall short of one.  Groups and pairs of more rows than a workgroup's smallest share.  And where the form that takes quantized
activations has the same bits."""
import numpy as np
import pytest

import oracle as fo
import test_gemv_groups as groups
from test_gpu_parity import assert_rows_close, bits, fa, make_weights, to_dev  # noqa: F401 (fa: the module's fixture)

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


# (every number of rows a workgroup takes in these two launches)
@pytest.mark.parametrize("kind,blocks,rows", [(fo.Q6_K, 2, (999, 251, 9)), (fo.Q6_K, 20, (999, 251, 9)), (fo.Q6_K, 5, (2047, 513, 9)), (fo.Q6_K, 5, (2999, 751, 9)),
                                              (fo.Q6_K, 20, (2999, 751, 9)), (fo.Q6_K, 5, (4095, 1025, 9)), (fo.Q6_K, 20, (4095, 1025, 9)), (fo.Q6_K, 5, (6999, 1751, 9)),
                                              (fo.Q6_K, 20, (6999, 1751, 9)), (fo.Q8_0, 9, (6999, 1751, 9))])
def test_larger_groups(fa, kind, blocks, rows):
    groups._group(fa, kind, 256 * blocks, rows)


@pytest.mark.parametrize("blocks,ffn", [(2, 992), (5, 1088), (20, 2272), (5, 2976)])
def test_larger_q6_k_gate_and_up(fa, blocks, ffn):
    groups.test_gate_up_and_swiglu_in_one_launch(fa, fo.Q6_K, blocks, ffn)


# Blocks at which one kernel's order of a row's sums is the other's, and lengths on either side
@pytest.mark.parametrize("kind,equal,others", [(fo.Q4_K, (1, 8, 9, 12, 15, 16, 65, 72), (17, 20, 21)), (fo.Q5_K, (1, 7, 8, 16, 32, 65, 72), (9, 12, 15, 17)),
                                               (fo.Q6_K, (1, 8, 9, 12, 15, 17, 19, 65, 72), (20, 24))])
def test_one_row_from_quantized_activations(fa, kind, equal, others):
    """frk_hip_gemv_q8k_dev and a one-row frk_hip_gemm_acts_dev against frk_hip_gemv_dev: the same bits, or the same integers in another
    order (a chain of at most nb + 6 additions of f32 terms no larger than the row's magnitudes in either)."""
    from frink_amd import synth
    for blocks in equal + others:
        for rows in (37, 2050):
            print("one row, quantized before", kind, rows, blocks, flush=True)
            cols = 256 * blocks
            data = make_weights(kind, 37, cols, seed=blocks)
            data = np.ascontiguousarray(np.resize(data.reshape(37, -1), (rows, data.size // 37))).reshape(-1)
            x = to_dev(synth.activations(blocks, 1, cols))
            w = fa.Weights.from_host(kind, data, rows, cols)
            want, got = w.gemv(x[0]).cpu().numpy(), w.gemv_q8k(fa.quantize_q8_k(x[0])).cpu().numpy()
            acts = fa.BatchActs(1, cols)
            acts.quantize(x)
            assert np.array_equal(bits(w.gemm_acts(acts).cpu().numpy()[0]), bits(got))
            if blocks in equal:
                assert np.array_equal(bits(got), bits(want)), (kind, rows, blocks)
            else:
                room = np.abs(x.cpu().numpy()).sum() * 3 * np.abs(fo.dequant(kind, data[:data.size // rows * 37])).max()
                assert np.abs(got - want).max() <= 2 * (blocks + 6) * 2.0 ** -24 * room
            acts.release()
            w.release()
