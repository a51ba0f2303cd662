"""The kernels of small K-quant batches beside gemm_k_rows_kernel, each at sizes that still go to it: row groups and tokens that are
not filled, the smallest and the larger of the kernel's shapes.  The launched kernel's name is checked on the CPU, the results on the GPU."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import fa, to_dev  # noqa: F401 (fa: the module's fixture)
from test_routes import kernels  # noqa: F401 (the module's fixture)

# (a launch's kernel, kind, rows, blocks, tokens)
SHAPES = [
    ("thin_span_q4_k_kernel<8>", fo.Q4_K, 45, 4, 7), ("thin_span_q4_k_kernel<8>", fo.Q4_K, 100, 12, 5), ("thin_span_q4_k_kernel<8>", fo.Q4_K, 33, 32, 8),
    ("thin_mfma_q4_k_kernel<1,4,false>", fo.Q4_K, 600, 80, 3), ("thin_mfma_q4_k_kernel<1,4,true>", fo.Q5_K, 601, 80, 2),
    ("thin_mfma_q4_k_kernel<2,4,false>", fo.Q4_K, 12301, 9, 3), ("thin_mfma_q4_k_kernel<2,4,true>", fo.Q5_K, 7140, 28, 2),
    ("thin_mfma_q4_k_kernel<2,8,false>", fo.Q4_K, 7141, 29, 5), ("thin_mfma_q4_k_kernel<2,8,true>", fo.Q5_K, 7139, 28, 7),
    ("thin_mfma_q4_k_kernel<4,4,false>", fo.Q4_K, 12300, 5, 4), ("thin_mfma_q4_k_kernel<4,4,true>", fo.Q5_K, 24600, 10, 2),
    ("thin_mfma_q4_k_kernel<4,8,false>", fo.Q4_K, 14300, 21, 5), ("thin_mfma_q4_k_kernel<4,8,true>", fo.Q5_K, 14301, 20, 6),
    ("thin_mfma_q4_k_kernel<4,16,false>", fo.Q4_K, 14300, 17, 9), ("thin_mfma_q4_k_kernel<4,16,true>", fo.Q5_K, 14300, 16, 15),
    ("thin_mfma_q4_k_kernel<8,4,false>", fo.Q4_K, 12333, 1, 3), ("thin_mfma_q4_k_kernel<8,4,true>", fo.Q5_K, 28560, 10, 3),
    ("thin_mfma_q4_k_kernel<8,8,false>", fo.Q4_K, 28561, 9, 5), ("thin_mfma_q4_k_kernel<8,8,true>", fo.Q5_K, 28560, 10, 8),
    ("thin_mfma_q4_k_kernel<8,16,false>", fo.Q4_K, 28560, 9, 16), ("thin_mfma_q4_k_kernel<8,16,true>", fo.Q5_K, 28560, 10, 11),
    ("thin_q4_k_kernel<16,2>", fo.Q4_K, 8201, 1, 2), ("thin_q4_k_kernel<32,2>", fo.Q4_K, 8200, 5, 2), ("thin_q4_k_kernel<64,2>", fo.Q4_K, 70, 20, 2),
    ("thin_q4_k_kernel<64,4>", fo.Q4_K, 15, 129, 9), ("thin_q6_k_kernel<16,2,1>", fo.Q6_K, 4101, 1, 2), ("thin_q6_k_kernel<32,2,1>", fo.Q6_K, 4100, 5, 2),
    ("thin_q6_k_kernel<64,2,1>", fo.Q6_K, 33, 20, 2), ("thin_q6_k_kernel<64,2,1>", fo.Q6_K, 17, 130, 5),
    ("thin_stream_q6_k_kernel", fo.Q6_K, 20, 2, 24), ("thin_stream_q6_k_kernel", fo.Q6_K, 200, 52, 11), ("thin_stream_q6_k_kernel", fo.Q6_K, 5001, 22, 6),
    ("thin_stream_q6_k_kernel", fo.Q6_K, 33, 60, 36), ("thin_stream_q6_k_kernel", fo.Q6_K, 901, 64, 12),
    ("gemm_q4_k_pipe_kernel<2,4,1>", fo.Q4_K, 65, 30, 17), ("gemm_q5_k_pipe_kernel<2,4,1>", fo.Q5_K, 40, 24, 20), ("batch_q6_k_pipe_kernel", fo.Q6_K, 1000, 79, 9),
    ("gemm_q4_k_pipe_kernel<2,4,1>", fo.Q4_K, 8200, 30, 31), ("gemm_q5_k_pipe_kernel<2,4,1>", fo.Q5_K, 8300, 27, 32), ("batch_q6_k_pipe_kernel", fo.Q6_K, 12300, 24, 25),
    ("batch_q6_k_pipe_kernel", fo.Q6_K, 4161, 48, 17),
]


def test_the_sizes_go_to_their_kernels(kernels):  # noqa: F811
    for shape, (rc, names) in zip(SHAPES, kernels([("gemm",) + s[1:] for s in SHAPES])):
        assert rc == 0 and shape[0] in names.split(), (shape, rc, names)


@pytest.mark.gpu
@pytest.mark.parametrize("kernel,kind,rows,blocks,batch", SHAPES)
def test_batches_match_exact_arithmetic(fa, kernel, kind, rows, blocks, batch):  # noqa: F811
    from bench import random_blocks
    from frink_amd import synth
    print("thin kernels", kernel, kind, rows, blocks, batch, flush=True)
    cols, some = 256 * blocks, min(rows, 211)  # (rows repeat: 211 divides no workgroup's share)
    base = random_blocks(kind, some, cols, seed=rows + cols)
    data = np.ascontiguousarray(np.resize(base.reshape(some, -1), (rows, base.size // some))).reshape(-1)
    x = synth.activations(batch, batch, cols, outlier_frac=0.01)
    w = fa.Weights.from_host(kind, data, rows, cols)
    got = w.gemm(to_dev(x)).cpu().numpy().astype(np.float64)
    w.release()
    a = np.empty((batch, cols), np.float64)
    for r in range(batch):
        q, d, _ = fo.quantize_q8_k(x[r])
        a[r] = (q.reshape(-1, 256).astype(np.float64) * d.astype(np.float64)[:, None]).ravel()
    wd = fo.dequant(kind, base).reshape(some, cols).astype(np.float64)
    # (the bound of test_batch_tiles.py: exact integers, a handful of f32 roundings a block and an addition for each, share and part)
    mag = np.abs(a) @ np.abs(wd).T
    if kind != fo.Q6_K:
        mag = mag + np.abs(a).sum(1)[:, None] * np.abs(wd).max(1)[None, :]
    room = (blocks + 24) * 2.0 ** -24 * mag
    at = np.arange(rows) % some
    assert (np.abs(got - (a @ wd.T)[:, at]) <= room[:, at]).all(), float((np.abs(got - (a @ wd.T)[:, at]) / room[:, at]).max())
