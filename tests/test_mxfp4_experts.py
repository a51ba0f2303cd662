"""MXFP4 experts on the block-scaled matrix cores (frk_gemm_mx.hip), at the edges of its tiles: rows, blocks a row, rows in
use of a tile, both workgroup sizes; and the activations whose Q8_0 scale leaves f16."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import _other_kind_blocks, fa, test_moe_ffn_with_experts_of_the_other_kinds, to_dev  # noqa: F401 (fa: a fixture)

_moe_case = test_moe_ffn_with_experts_of_the_other_kinds
del test_moe_ffn_with_experts_of_the_other_kinds  # (collected in its own file)


def _case(fa, counts, rows_g, cols, x, seed):
    n_groups = len(counts)
    off = np.zeros(n_groups + 1, np.int32)
    off[1:] = np.cumsum(counts)
    data = _other_kind_blocks(fo.MXFP4, n_groups * rows_g, cols, seed=seed)
    blk = data.reshape(-1, 17)
    blk[:, 0] = 104 + blk[:, 0] % 40
    w = fa.Weights.from_host(fo.MXFP4, data, n_groups * rows_g, cols)
    got = fa.gemm_grouped(w, n_groups, to_dev(off), to_dev(x)).cpu().numpy()
    w.release()
    return off, data.reshape(n_groups, -1), got


@pytest.mark.gpu
@pytest.mark.parametrize("rows_g,cols,counts", [
    (1, 32, [1, 64]), (63, 96, [0, 33, 2]), (65, 128, [32, 31, 65]), (257, 160, [64, 5]), (72, 544, [97, 1]),
    (512, 1056, [40]), (1100, 160, [3, 0, 34] * 30),
    # (rows from 384 columns on are frk_gemm_mx.hip's: three quads of blocks, and one to four blocks of a last one; the last:
    # eight wavefronts a workgroup, three workgroups a tile)
    (1, 384, [1, 64]), (63, 416, [0, 33, 2]), (65, 448, [32, 31, 65]), (257, 480, [64, 5]), (72, 512, [97, 1]),
    (1100, 416, [3, 0, 34] * 30),
])
def test_grouped_gemm_at_the_edges_of_its_tiles(fa, rows_g, cols, counts):
    from frink_amd import synth
    print("mxfp4 experts", rows_g, cols, len(counts), flush=True)
    pairs = sum(counts)
    x = synth.activations(71, pairs, cols, outlier_frac=0.01)
    off, per, got = _case(fa, counts, rows_g, cols, x, seed=rows_g + cols)
    # Q8_0 activations in exact arithmetic.  A matrix-core step sums 64 exact products within 8 units in the last place
    # of its largest (6.2 seen), eight steps in a row to a running sum of 128 columns, then one addition each.
    xb = x.reshape(pairs, cols // 32, 32)
    amax = np.abs(xb).max(axis=2)
    inv = np.where(amax != 0, np.float32(127) / np.where(amax != 0, amax, 1), 0).astype(np.float32)
    q = np.clip(np.rint(xb * inv[:, :, None]), -127, 127).astype(np.float64)
    a = (q * (amax / np.float32(127)).astype(np.float16).astype(np.float64)[:, :, None]).reshape(pairs, cols)
    for g in range(len(counts)):
        s = slice(int(off[g]), int(off[g + 1]))
        wd = fo.dequant(fo.MXFP4, per[g]).reshape(rows_g, cols).astype(np.float64)
        room = (64 + cols // 128 + 1) * 2.0 ** -24 * (np.abs(a[s]) @ np.abs(wd).T)
        assert (np.abs(got[s] - a[s] @ wd.T) <= room).all(), g


@pytest.mark.gpu
@pytest.mark.parametrize("cols,scale", [(384, 1.0), (416, 2.0 ** -20), (1056, 6.0e4)])  # (the middle one: subnormal f16 scales)
def test_digits_of_every_activation_are_exact(fa, cols, scale):
    """A weight row that picks one column returns that activation's quant times scale: its digits' sum, no rounding."""
    rng = np.random.default_rng(cols)
    x = (rng.standard_normal((96, cols)) * scale * 2.0 ** rng.integers(-3, 4, (96, 1))).astype(np.float32)
    x[0], x[1] = scale * 127, -scale * 127 * 2047 / 2048  # all ends, and all bits of a scale
    x[2, ::3] = 0
    x[3, 32:64] = 0
    blk = np.zeros((cols, cols // 32, 17), np.uint8)
    blk[:, :, 0] = 127
    c = np.arange(cols)
    blk[c, c // 32, 1 + c % 16] = np.where(c % 32 < 16, 0x02, 0x20)  # E2M1 one
    w = fa.Weights.from_host(fo.MXFP4, blk.reshape(-1), cols, cols)
    got = fa.gemm_grouped(w, 1, to_dev(np.array([0, 96], np.int32)), to_dev(x)).cpu().numpy()
    w.release()
    xb = x.reshape(96, cols // 32, 32)
    amax = np.abs(xb).max(axis=2)
    inv = np.where(amax != 0, np.float32(127) / np.where(amax != 0, amax, 1), 0).astype(np.float32)
    q = np.clip(np.rint(xb * inv[:, :, None]), -127, 127)
    a = q * (amax / np.float32(127)).astype(np.float16).astype(np.float32)[:, :, None]
    assert np.array_equal(got, a.reshape(96, cols).astype(np.float32))


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [64, 96, 352])
def test_short_rows_round_once_a_block(fa, cols):
    """Below 384 columns a block's sum is an exact integer with one rounding behind it, added in the blocks' order."""
    from frink_amd import synth
    rows_g, counts = 80, [70, 50]
    x = synth.activations(77, sum(counts), cols, outlier_frac=0.02)
    off, per, got = _case(fa, counts, rows_g, cols, x, seed=cols)
    xb = x.reshape(-1, cols // 32, 32)
    amax = np.abs(xb).max(axis=2)
    inv = np.where(amax != 0, np.float32(127) / np.where(amax != 0, amax, 1), 0).astype(np.float32)
    q = np.clip(np.rint(xb * inv[:, :, None]), -127, 127).astype(np.float64)
    a = q * (amax / np.float32(127)).astype(np.float16).astype(np.float64)[:, :, None]
    for g in range(len(counts)):
        s = slice(int(off[g]), int(off[g + 1]))
        wd = fo.dequant(fo.MXFP4, per[g]).reshape(rows_g, cols // 32, 32).astype(np.float64)
        running = np.cumsum(np.einsum("tbi,rbi->trb", a[s], wd), axis=2)
        # half a unit in the last place of every running sum, and of what the roundings before have made of it
        room = 2.0 ** -24 * (np.abs(running).sum(axis=2) * (1 + 2.0 ** -20) + cols // 32 * 2.0 ** -24 * np.abs(running).max(axis=2))
        assert (np.abs(got[s] - running[:, :, -1]) <= room).all(), g


@pytest.mark.gpu
def test_activations_whose_scale_leaves_f16(fa):
    """An infinite value empties its block (0 times an infinite scale: NaN), one above 8.3e6 makes the results infinite
    with its block's sign, a NaN counts as zero; a tiny block's scale is an f16 subnormal; the other rows are untouched."""
    rng = np.random.default_rng(5)
    x = rng.standard_normal((40, 96)).astype(np.float32)
    x[3, 40] = np.inf
    x[7, 10] = 2.0e7
    x[9, 50] = np.nan
    x[11, :32] *= 1e-5
    x[12] = 0.0
    off, per, got = _case(fa, [40], 70, 96, x, seed=9)
    want = fo.gemm(fo.MXFP4, per[0], 70, 96, x, fo.INT_DOT)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(got[3]).all()
    assert np.isinf(got[7]).any() and np.array_equal(np.isinf(got), np.isinf(want))
    inf = np.isinf(want)
    assert np.array_equal(np.sign(got[inf]), np.sign(want[inf]))
    fine = [r for r in range(40) if r not in (3, 7)]
    assert (np.abs(got[fine] - want[fine]).max(axis=1) <= 1e-5 * np.abs(want[fine]).max(axis=1)).all()


@pytest.mark.gpu
def test_rows_with_several_blocks_whose_scale_leaves_f16(fa):
    """Every such block adds an infinity of its own: two that agree stay infinite, two that differ give NaN, as does one
    whose integer sum is zero beside one whose sum is not."""
    cols, rows_g = 416, 70
    rng = np.random.default_rng(11)
    x = rng.standard_normal((70, cols)).astype(np.float32)
    x[3, [10, 200]] = 2.0e7
    x[7, [10, 200, 415]] = 1.0e8, -3.0e7, 2.0e8
    x[40, 64:96] = 9.0e6 * rng.standard_normal(32)
    x[40, 96] = -1.0e9
    x[66, [0, 33]] = np.inf, 2.0e7
    x[9, 50] = np.nan       # (counts as zero)
    x[11, :32] *= 1e-5      # (an f16 subnormal scale)
    x[12] = 0.0
    off, per, got = _case(fa, [33, 37], rows_g, cols, x, seed=21)
    large = [3, 7, 40, 66]
    for g in range(2):
        s = slice(int(off[g]), int(off[g + 1]))
        want = fo.gemm(fo.MXFP4, per[g], rows_g, cols, x[s], fo.INT_DOT)
        assert np.array_equal(np.isnan(got[s]), np.isnan(want)) and np.array_equal(np.isinf(got[s]), np.isinf(want))
        inf = np.isinf(want)
        assert np.array_equal(np.sign(got[s][inf]), np.sign(want[inf]))
        fine = [r for r in range(want.shape[0]) if r + s.start not in large]
        assert (np.abs(got[s][fine] - want[fine]).max(axis=1) <= 1e-5 * np.abs(want[fine]).max(axis=1)).all()
    for r in (3, 7, 40):  # (rows with both outcomes)
        assert np.isnan(got[r]).any() and np.isinf(got[r]).any()
    assert np.isnan(got[66]).all()


@pytest.mark.gpu
def test_moe_layer_whose_intermediates_leave_f16(fa):
    """The same between gate/up and the down projection: a layer of a few tokens runs a job per pair, a batch the grouped
    kernels, and a token's results are of the same kind in both."""
    import torch
    n_experts, hidden, ffn, batch = 4, 416, 448, 40
    rng = np.random.default_rng(12)
    ws = []
    for i, (rows, cols) in enumerate(((ffn, hidden), (ffn, hidden), (hidden, ffn))):
        data = _other_kind_blocks(fo.MXFP4, n_experts * rows, cols, seed=30 + i)
        data.reshape(-1, 17)[:, 0] = 118 + data.reshape(-1, 17)[:, 0] % 4
        ws.append(fa.Weights.from_host(fo.MXFP4, data, n_experts * rows, cols))
    x = rng.standard_normal((batch, hidden)).astype(np.float32)
    x[5] *= 2.0e4       # finite gate and up, products past 8.3e6 in many blocks
    x[9, [3, 300]] = 2.0e7   # infinite gate and up
    ids = to_dev(rng.integers(0, n_experts, (batch, 1)).astype(np.int32))
    weights = torch.ones((batch, 1), dtype=torch.float32, device="cuda")
    xd = to_dev(x)
    got = fa.moe_ffn(*ws, n_experts, xd, ids, weights).cpu().numpy()
    want = np.concatenate([fa.moe_ffn(*ws, n_experts, xd[i:i + 8].contiguous(), ids[i:i + 8].contiguous(), weights[i:i + 8].contiguous()).cpu().numpy()
                           for i in range(0, batch, 8)])
    assert not np.isfinite(want[5]).all() and not np.isfinite(want[9]).all()
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    inf = np.isinf(want)
    assert np.array_equal(np.sign(got[inf]), np.sign(want[inf]))
    fine = [r for r in range(batch) if r not in (5, 9)]
    # (an intermediate's last bit now and then moves a quant of the down projection's input to the next level)
    assert (np.abs(got[fine] - want[fine]).max(axis=1) <= 2e-3 * np.abs(want[fine]).max(axis=1)).all()
    for w in ws:
        w.release()


@pytest.mark.gpu
@pytest.mark.parametrize("n_experts,k,hidden,ffn,batch", [(64, 2, 160, 1056, 40), (3, 2, 544, 288, 33), (8, 2, 288, 544, 16), (16, 2, 96, 160, 15),
                                                            (64, 2, 416, 1056, 40), (3, 2, 544, 416, 33), (8, 2, 480, 544, 16)])
def test_moe_layer_at_the_edges_of_its_tiles(fa, n_experts, k, hidden, ffn, batch):
    _moe_case(fa, fo.MXFP4, fo.MXFP4, n_experts, k, hidden, ffn, batch)


@pytest.mark.gpu
@pytest.mark.parametrize("rows_g,cols,counts", [
    (1500, 416, [96, 97, 65, 64, 128, 192, 193, 0, 1] * 3),  # four wavefronts a workgroup, one to three halves, last tiles of a row
    (4097, 416, [96, 65, 33, 1, 97, 32, 64, 200] * 4),  # nine workgroups a tile, an XCD's last round of jobs cut in two
])
def test_tiles_of_96_rows(fa, rows_g, cols, counts):
    test_grouped_gemm_at_the_edges_of_its_tiles(fa, rows_g, cols, counts)


@pytest.mark.gpu
@pytest.mark.parametrize("rows_g,cols,counts", [
    (1500, 416, [96, 97, 65, 64, 128, 192, 193, 0, 1] * 3),
    (4097, 416, [96, 65, 33, 1, 97, 32, 64, 200] * 4),  # among the jobs cut in two: tiles of one and two halves
    (8190, 384, [96] * 9),                               # cut in two: all jobs of the XCDs with one tile, of three halves
])
def test_rows_whose_scale_leaves_f16_in_tiles_of_96(fa, rows_g, cols, counts):
    """Infinite results where and with the signs the oracle has them, in every half of a tile; the other rows keep their bits."""
    print("mxfp4 infinite rows", rows_g, cols, len(counts), flush=True)
    rng = np.random.default_rng(rows_g)
    x = rng.standard_normal((sum(counts), cols)).astype(np.float32)
    large = x.copy()
    off = np.concatenate(([0], np.cumsum(counts)))
    rows = [sorted({r % n for r in (5, 31, 40, 63, 70, 95, n - 1)}) if n else [] for n in counts]
    for g, picked in enumerate(rows):
        for i, r in enumerate(picked):
            large[off[g] + r, 7 * i + 1] = 2.0e7
            large[off[g] + r, 370 - 9 * i] = (3.0e7, -3.0e7, 1.0, np.inf)[(g + i) % 4]
    _, per, finite = _case(fa, counts, rows_g, cols, x, seed=41)
    _, _, got = _case(fa, counts, rows_g, cols, large, seed=41)
    untouched = np.ones(len(x), bool)
    for g, picked in enumerate(rows):
        if not picked:
            continue
        at = off[g] + np.array(picked)
        untouched[at] = False
        want = fo.gemm(fo.MXFP4, per[g], rows_g, cols, large[at], fo.INT_DOT)
        assert not np.isfinite(want).any()
        assert np.array_equal(np.isnan(got[at]), np.isnan(want)), g
        assert np.array_equal(np.sign(got[at][np.isinf(want)]), np.sign(want[np.isinf(want)])), g
    assert np.array_equal(got[untouched].view(np.uint32), finite[untouched].view(np.uint32))


@pytest.mark.parametrize("pairs,groups,rows,glu,tile", [
    (832, 8, 2048, True, 64), (896, 8, 2880, True, 64), (1728, 16, 1536, True, 64),  # two tiles an expert, one round of the chip
    (2776, 8, 1088, True, 64),  # two rounds of four wavefronts' workgroups with either tile
    (1000, 16, 1536, True, 96), (2048, 32, 2880, True, 96), (2400, 8, 2880, True, 96),
    (2508, 27, 1500, False, 96), (2352, 32, 4097, False, 96), (840, 9, 4064, True, 96), (864, 9, 8190, False, 96),  # the tests of such tiles here
])
def test_tiles_of_96_rows_where_those_of_64_do_not_fit_the_chip_at_once(pairs, groups, rows, glu, tile):
    import ctypes as C

    import frink_amd
    f = frink_amd.lib()._ZN3frk7mx_tileEmmmb  # frk::mx_tile
    f.restype, f.argtypes = C.c_int, [C.c_size_t] * 3 + [C.c_bool]
    assert f(pairs, groups, rows, glu) == tile


@pytest.mark.gpu
def test_layer_whose_last_round_of_jobs_is_cut_in_two(fa):
    """Sixteen workgroups a tile: the XCDs with one tile (or three) cut a round of sixteen jobs in two, tiles of one to
    three halves among them, the last 32 rows missing."""
    _moe_case(fa, fo.MXFP4, fo.MXFP4, 9, 2, 416, 4064, 420)


def test_no_result_of_the_matrix_core_is_read_too_soon(tmp_path):
    import isa_mfma_lint
    from test_isa_waits import _assembly
    asm = _assembly(tmp_path, "frk_gemm_mx.hip")
    assert "v_mfma_scale_f32_32x32x64_f8f6f4" in asm
    assert isa_mfma_lint.violations(asm) == []
