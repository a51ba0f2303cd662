"""The grouped K-quant GEMM's items of 128 weight rows (frk_gemm.hip, stream_gemm): last items of 1, 127 and 1 + 128 rows, one
to three blocks a row (a workgroup's first steps are its last), tiles with and without a second half, lists longer than
the items that two workgroups a CU hold."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import _grouped_case, _grouped_oracle, assert_rows_close, fa, to_dev  # noqa: F401 (fa: the module's fixture)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [fo.Q4_K, fo.Q6_K])
@pytest.mark.parametrize("rows_g,cols,counts", [
    (1, 256, [1]), (127, 512, [33, 2]), (129, 256, [64, 0, 1]), (257, 768, [40, 5, 65]), (1100, 256, [3] * 70),
])
def test_items_of_128_rows(fa, kind, rows_g, cols, counts):
    print("grouped stream", kind, rows_g, cols, flush=True)
    for with_gather in (True, False):
        data, x, off, gather, pairs = _grouped_case(kind, len(counts), rows_g, cols, counts, 50, rows_g + cols + kind, with_gather)
        w = fa.Weights.from_host(kind, data, len(counts) * rows_g, cols)
        got = fa.gemm_grouped(w, len(counts), to_dev(off), to_dev(x), to_dev(gather) if with_gather else None).cpu().numpy()
        assert_rows_close(got, _grouped_oracle(kind, data, len(counts), rows_g, cols, x, off, gather), "grouped stream")
        w.release()


@pytest.mark.gpu
def test_more_items_than_the_workgroups_hold(fa):
    """15360 items of one block, where 512 workgroups hold 28 each: the same bits as in two calls of half the groups."""
    import torch
    n, rows_g, cols = 1024, 1920, 256
    print("grouped stream, 15360 items", flush=True)
    gen = torch.Generator("cuda")
    gen.manual_seed(3)
    blocks = torch.randint(0, 256, (n * rows_g, 144), generator=gen, device="cuda", dtype=torch.uint8)
    blocks[:, 1], blocks[:, 3] = 0x12, 0x14  # f16 scales of about 1e-3
    x = torch.randn((n, cols), generator=gen, device="cuda")

    def run(g0, g1):
        w = fa.Weights.from_device(fo.Q4_K, blocks[g0 * rows_g:g1 * rows_g].reshape(-1).contiguous(), (g1 - g0) * rows_g, cols)
        y = fa.gemm_grouped(w, g1 - g0, torch.arange(g1 - g0 + 1, dtype=torch.int32, device="cuda"), x[g0:g1].contiguous()).cpu().numpy()
        w.release()
        return y

    assert np.array_equal(run(0, n).view(np.uint32), np.concatenate([run(0, n // 2), run(n // 2, n)]).view(np.uint32))
