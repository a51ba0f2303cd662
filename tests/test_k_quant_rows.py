"""K-quant batches of 2 to 32 rows, and more of small matrices, on sixteen-row workgroups (gemm_k_rows_kernel, frk_gemm_rows.hip): rows that fill no
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
          (fo.Q6_K, 2062, 9984, 30), (fo.Q5_K, 2570, 14336, 32)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", SHAPES)
def test_batches_match_exact_arithmetic(fa, kind, rows, cols, batch):
    _check(fa, kind, rows, cols, batch)


# (several tiles of tokens: one and sixteen rows of the last, whole ones; both sides of the line to the pipelined GEMM)
TILES = [(fo.Q4_K, 17, 256, 33), (fo.Q4_K, 1101, 2048, 103), (fo.Q4_K, 47, 9216, 64), (fo.Q4_K, 1319, 9216, 63), (fo.Q4_K, 1318, 9216, 128), (fo.Q5_K, 15, 1280, 48),
         (fo.Q5_K, 1782, 3072, 65), (fo.Q5_K, 33, 17152, 40), (fo.Q5_K, 4100, 512, 81), (fo.Q6_K, 1, 768, 34), (fo.Q6_K, 600, 3584, 511), (fo.Q6_K, 601, 3584, 512),
         (fo.Q6_K, 31, 8448, 96)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", TILES)
def test_several_tiles_match_exact_arithmetic(fa, kind, rows, cols, batch):
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


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", [TILES[i] for i in (0, 1, 6, 7, 12)])
def test_every_entry_point_has_the_same_bits_over_several_tiles(fa, kind, rows, cols, batch):
    import torch
    from frink_amd import synth
    print("k-quant rows, tiles", kind, rows, cols, batch, flush=True)
    w = fa.Weights.from_host(kind, make_weights(kind, rows, cols, seed=rows), rows, cols)
    x = to_dev(synth.activations(batch, batch, cols))
    room = torch.full((batch * rows + 128,), 7.0, device="cuda")
    y = room[64:-64].view(batch, rows)
    w.gemm(x, out=y)
    want = bits(y.cpu().numpy())
    assert (room[:64] == 7.0).all() and (room[-64:] == 7.0).all()
    acts = fa.BatchActs(batch, cols)
    acts.quantize(x)
    assert np.array_equal(bits(w.gemm_acts(acts).cpu().numpy()), want)
    for y in fa.gemm_pair(w, w, x):
        assert np.array_equal(bits(y.cpu().numpy()), want)
    y = torch.full((batch, rows), float("nan"), device="cuda")
    w.gemm_noalloc(x, y)
    assert np.array_equal(bits(y.cpu().numpy()), want)
    for t in range(0, batch, 32):  # (a tile of its own: the tokens of a batch of 2 to 32 where those are this kernel's too)
        if min(batch - t, 32) > 1 and rows <= 2048 and cols < 19 * 256:
            assert np.array_equal(bits(w.gemm(x[t:t + 32].contiguous()).cpu().numpy()), want[t:t + 32])
    w.release()


# (the pipelined GEMM's batches whose tiles come from the same quantizer, rows past the batch cleared: one row of an octet and all of it, and both
# sides of the 400 records from where a record is a workgroup's)
CLEARED = [(fo.Q4_K, 2000, 9216, 33), (fo.Q4_K, 2000, 9216, 40), (fo.Q5_K, 3000, 9216, 41), (fo.Q6_K, 3300, 9216, 63), (fo.Q4_K, 400, 9216, 352),
           (fo.Q4_K, 400, 9216, 353)]


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", CLEARED)
def test_pipelined_batches_from_the_lanes_match_exact_arithmetic(fa, kind, rows, cols, batch):
    _check(fa, kind, rows, cols, batch)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", CLEARED)
def test_rows_of_an_earlier_batch_leave_the_tiles(fa, kind, rows, cols, batch):
    from frink_amd import synth
    print("octets after a larger batch", kind, rows, cols, batch, flush=True)
    w = fa.Weights.from_host(kind, make_weights(kind, rows, cols, seed=rows), rows, cols)
    x = to_dev(synth.activations(batch, batch, cols))
    want = bits(w.gemm(x).cpu().numpy())
    acts = fa.BatchActs(batch + 31, cols)
    large = to_dev(synth.activations(batch, batch + 31, cols))
    large[batch:] = float("inf")  # (scales that are not finite in the rows that the next batch does not have)
    acts.quantize(large)
    acts.quantize(x)
    assert np.array_equal(bits(w.gemm_acts(acts).cpu().numpy()), want)
    w.release()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [fo.Q4_K, fo.Q5_K])
@pytest.mark.parametrize("blocks", [1, 2, 3, 15, 16, 17, 31])  # (one block, a pair, a half pair at the end; shares of one and two pairs; more are refused from 9 rows on)
def test_plain_rows_through_lds(fa, kind, blocks):
    """From Q8_K rows as they are the same bits as from tiles, whatever tokens of the sixteen are in use."""
    from frink_amd import synth
    rows, cols = 35, 256 * blocks
    w = fa.Weights.from_host(kind, make_weights(kind, rows, cols, seed=blocks), rows, cols)
    for batch in (3, 5, 8, 11, 13, 16):
        print("plain rows", kind, blocks, batch, flush=True)
        x = to_dev(synth.activations(batch, batch, cols, outlier_frac=0.01))
        got = w.gemm_q8k(fa.quantize_q8_k(x.reshape(-1)), batch)
        assert np.array_equal(bits(got.cpu().numpy()), bits(w.gemm(x).cpu().numpy())), batch
    w.release()
