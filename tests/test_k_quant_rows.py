"""K-quant batches of 2 to 32 rows on sixteen-row workgroups (gemm_k_rows_kernel, frk_gemm_rows.hip): rows that fill no
workgroup, odd numbers of blocks and of pairs a wavefront, one and two tiles of tokens; every entry point the same bits."""
import numpy as np
import pytest

import oracle as fo
from test_batch_tiles import _check
from test_gpu_parity import bits, fa, make_weights, to_dev  # noqa: F401 (fa: the module's fixture)

# (one and two tokens' tiles, their edges; 1 .. 9 and 17 .. 34 pairs of blocks over at most eight wavefronts, the last pair whole and
# half; one row, one short of a workgroup, one and a part, several)
SHAPES = [(fo.Q4_K, 15, 2304, 3), (fo.Q4_K, 17, 256, 16), (fo.Q4_K, 33, 1280, 17), (fo.Q4_K, 1, 4864, 32), (fo.Q4_K, 1030, 11008, 8),
          (fo.Q4_K, 2100, 8192, 31), (fo.Q4_K, 100, 8448, 9), (fo.Q5_K, 1, 256, 2), (fo.Q5_K, 31, 512, 15), (fo.Q5_K, 16, 4864, 17), (fo.Q5_K, 50, 17152, 5),
          (fo.Q5_K, 2070, 14336, 32), (fo.Q6_K, 1, 256, 3), (fo.Q6_K, 18, 768, 17), (fo.Q6_K, 47, 4096, 16), (fo.Q6_K, 16, 4352, 32), (fo.Q6_K, 35, 17152, 9),
          (fo.Q6_K, 2062, 9984, 30)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", SHAPES)
def test_batches_match_exact_arithmetic(fa, kind, rows, cols, batch):
    _check(fa, kind, rows, cols, batch)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", [SHAPES[i] for i in (0, 3, 7, 8, 13, 15)])
def test_every_entry_point_has_the_same_bits(fa, kind, rows, cols, batch):
    import torch
    from frink_amd import synth
    print("k-quant rows", kind, rows, cols, batch, flush=True)
    w = fa.Weights.from_host(kind, make_weights(kind, rows, cols, seed=rows), rows, cols)
    x = to_dev(synth.activations(batch, batch, cols))
    want = bits(w.gemm(x).cpu().numpy())
    assert np.array_equal(bits(w.gemm_q8k(fa.quantize_q8_k(x.reshape(-1)), batch).cpu().numpy()), want)
    acts = fa.BatchActs(batch, cols)
    acts.quantize(x)
    assert np.array_equal(bits(w.gemm_acts(acts).cpu().numpy()), want)
    for y in fa.gemm_pair(w, w, x):
        assert np.array_equal(bits(y.cpu().numpy()), want)
    y = torch.full((batch, rows), float("nan"), device="cuda")
    w.gemm_noalloc(x, y)
    assert np.array_equal(bits(y.cpu().numpy()), want)
    w.release()


def test_compiled_kernels_keep_the_waits(tmp_path):
    import isa_mfma_lint
    import isa_wait_lint
    from test_isa_waits import _assembly
    asm = _assembly(tmp_path, "frk_gemm_rows.hip")
    assert isa_mfma_lint.violations(asm) == []
    names = isa_wait_lint.kernels(asm)
    assert sum("gemm_k_rows" in k for k in names) == 10 and len(names) == 11, names  # (and the batch's quantizer)
    for k in names:
        assert isa_wait_lint.violations(asm, k) == [], k
