"""The matrix-core kernels at the edges of their tiles and splits, on arbitrary block bytes (every scale and code)."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import fa, to_dev  # noqa: F401 (fa: the module's fixture)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,batch", [
    (33, 512, 65),        # one row group and one token past a tile, two blocks a row
    (257, 2816, 130),     # a row past a large tile, eleven blocks: splits of unequal length
    (129, 16384, 70),     # 64 blocks split over eight workgroups
    (4130, 1024, 700),    # large tiles, the last of both kinds partly filled
    (1, 768, 97),
])
@pytest.mark.parametrize("kind", [fo.Q4_K, fo.Q5_K, fo.Q6_K])
def test_pipelined_gemm_at_the_edges_of_its_tiles(fa, kind, rows, cols, batch):
    from bench import random_blocks
    from frink_amd import synth
    data = random_blocks(kind, rows, cols, seed=rows + kind)
    x = synth.activations(31 + batch, batch, cols, outlier_frac=0.01)
    w = fa.Weights.from_host(kind, data, rows, cols)
    got = w.gemm(to_dev(x)).cpu().numpy().astype(np.float64)
    q, d, _ = fo.quantize_q8_k(x.reshape(-1))
    a = (q.reshape(-1, 256).astype(np.float64) * d.reshape(-1, 1).astype(np.float64)).reshape(batch, cols)
    wd = fo.dequant(kind, data).reshape(rows, cols).astype(np.float64)
    # Per block an output gains d_a * (d * S1 - dmin * S2): integers exact (S1 rounded once to f32), up to eight f32
    # roundings, then one per block in the sum; every rounding is of a number no larger than |W| |x| with the two terms
    # of Q4_K and Q5_K, whose difference the weight is, taken apart.  |d * sc * q| and |dmin * m| are each below the sum
    # of the largest weight of their row and twice its largest offset, hence the row's largest |w| times sum |x|.
    room = np.abs(a).sum(axis=1)[:, None] * (3.0 * np.abs(wd).max(axis=1))[None, :]
    assert (np.abs(got - a @ wd.T) <= (cols // 256 + 9) * 2.0 ** -24 * room).all()
    w.release()


@pytest.mark.parametrize("kind,rows,cols", [
    (fo.Q4_K, 40, 8448),     # rows past 32 blocks: the matrix cores from 9 rows on
    (fo.Q4_K, 4104, 6144),   # 24 blocks, past one workgroup a CU: from 9
    (fo.Q5_K, 72, 8192),     # 32 blocks: from 9
    (fo.Q5_K, 264, 4096),    # 16 blocks of few rows: from 17
    (fo.Q6_K, 4104, 8448),   # large, an odd number of blocks: from 9
    (fo.Q6_K, 8200, 4352),   # the same with 17 blocks, whose batches have no tiles below 17 rows: from 17
    # (gemm_k_rows_kernel has those above on both sides of 9, the third and the last two of 17; on the tiles from 9, 9 and 17 on:)
    (fo.Q4_K, 72, 12288), (fo.Q5_K, 72, 12288), (fo.Q6_K, 1300, 12544),
])
def test_batches_around_the_step_from_thin_to_tiled(fa, kind, rows, cols):
    """Both sides of the batch size at which a matrix changes kernels, against 64-bit sums of the same quantized
    operands; the activations' two forms come out of one launch, and a product over them is the plain call's bit for bit."""
    from bench import random_blocks
    from frink_amd import synth
    data = random_blocks(kind, rows, cols, seed=rows + kind)
    wd = fo.dequant(kind, data).reshape(rows, cols).astype(np.float64)
    w = fa.Weights.from_host(kind, data, rows, cols)
    acts = fa.BatchActs(33, cols)
    for batch in (8, 9, 16, 17, 33):
        x = synth.activations(7 + batch, batch, cols, outlier_frac=0.01)
        xd = to_dev(x)
        y = w.gemm(xd).cpu().numpy()
        assert np.array_equal(w.gemm_acts(acts.quantize(xd)).cpu().numpy().view(np.uint32), y.view(np.uint32)), batch
        q, d, _ = fo.quantize_q8_k(x.reshape(-1))
        a = (q.reshape(-1, 256).astype(np.float64) * d.reshape(-1, 1).astype(np.float64)).reshape(batch, cols)
        # (the bound of the test above, whose kernel adds a block at a time; the thin kernels' chains are no longer)
        room = np.abs(a).sum(axis=1)[:, None] * (3.0 * np.abs(wd).max(axis=1))[None, :]
        assert (np.abs(y.astype(np.float64) - a @ wd.T) <= (cols // 256 + 9) * 2.0 ** -24 * room).all(), batch
    acts.release()
    w.release()


@pytest.mark.parametrize("kind,rows,cols", [(fo.Q4_K, 640, 9728), (fo.Q5_K, 640, 8192), (fo.Q6_K, 4104, 8448), (fo.Q4_K, 640, 12288), (fo.Q5_K, 640, 12288),
                                            (fo.Q6_K, 1000, 20224)])
def test_a_batch_past_the_thin_kernels_is_no_further_from_64_bit_sums(fa, kind, rows, cols):
    """Eight rows run on sixteen-row workgroups and nine (of the last three sizes) on tiles whose parts are added by a second launch:
    the larger batch must not be less precise.  The
    2-norms of thousands of independent errors are within a few percent of their expectation, hence the tenth."""
    from frink_amd import synth
    # (encoded rows, whose offsets and scaled codes nearly cancel as a checkpoint's do)
    distinct = fo.encode_matrix(kind, synth.weights(5 + kind, 160, cols))
    data = np.resize(distinct.reshape(160, -1), (rows, distinct.size // 160)).reshape(-1)
    x = synth.activations(9, 9, cols, outlier_frac=0.002)
    q, d, _ = fo.quantize_q8_k(x.reshape(-1))
    a = (q.reshape(-1, 256).astype(np.float64) * d.reshape(-1, 1).astype(np.float64)).reshape(9, cols)
    exact = a @ fo.dequant(kind, distinct).reshape(160, cols).astype(np.float64).T
    w = fa.Weights.from_host(kind, data, rows, cols)
    nine = np.linalg.norm(w.gemm(to_dev(x)).cpu().numpy()[:8, :160] - exact[:8])
    eight = np.linalg.norm(w.gemm(to_dev(x[:8])).cpu().numpy()[:, :160] - exact[:8])
    w.release()
    assert nine <= 1.1 * eight, (nine, eight)
