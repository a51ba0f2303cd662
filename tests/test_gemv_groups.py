"""Matrices of one kind in one decode launch (frk_hip_gemv_multi_dev): rows that no workgroup's share divides, one row, one to
five matrices (four a launch), rows of one block to more than the column form's, every output between guards."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import assert_rows_close, bits, fa, make_weights, to_dev  # noqa: F401 (fa: the module's fixture)

GUARD = 64


def _group(fa, kind, cols, rows):
    import torch
    from frink_amd import synth
    data = [make_weights(kind, r, cols, seed=3 * cols + r + i) for i, r in enumerate(rows)]
    x = synth.activations(cols + kind, 1, cols, outlier_frac=0.01)[0]
    ws = [fa.Weights.from_host(kind, d, r, cols) for d, r in zip(data, rows)]
    room = torch.full((sum(rows) + GUARD * (len(rows) + 1),), 7.0, device="cuda")
    ys, at = [], GUARD
    for r in rows:
        ys.append(room[at:at + r])
        at += r + GUARD
    fa.gemv_multi(ws, to_dev(x), outs=ys)
    all_of = room.cpu().numpy()
    at = 0
    for r in list(rows) + [0]:
        assert (all_of[at:at + GUARD] == 7.0).all(), "a guard was overwritten"
        at += GUARD + r
    for w, d, y, r in zip(ws, data, ys, rows):
        got = y.cpu().numpy()
        assert_rows_close(got[None], fo.gemv(kind, d, r, cols, x, fo.F32_DOT if kind == fo.Q8_0 else fo.INT_DOT)[None], "group kind %d %dx%d" % (kind, r, cols))
        if kind in (fo.Q6_K, fo.Q8_0):  # (the same kernel on its own)
            assert np.array_equal(bits(got), bits(w.gemv(to_dev(x)).cpu().numpy()))
        else:
            assert_rows_close(w.gemv(to_dev(x)).cpu().numpy()[None], got[None], "alone, kind %d %dx%d" % (kind, r, cols))
        w.release()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [fo.Q4_K, fo.Q5_K, fo.Q6_K, fo.Q8_0])
@pytest.mark.parametrize("blocks,rows", [
    (1, (3, 1)), (3, (33, 9, 17)), (8, (64, 8, 8)), (8, (65, 7)), (9, (40, 1, 130)), (12, (7,)), (15, (257, 31, 5, 90, 12)), (16, (128, 4, 20)),
    (16, (129, 3)), (17, (100, 50, 50)), (20, (15,)), (24, (2049, 9)), (32, (66, 34, 2)), (40, (70, 30)), (64, (21, 11)), (66, (9, 4)),
])
def test_groups_of_a_kind(fa, kind, blocks, rows):
    print("gemv group", kind, blocks, rows, flush=True)
    _group(fa, kind, 256 * blocks, rows)


@pytest.mark.gpu
def test_neighbours_of_a_kind_in_a_mixed_list(fa):
    """Q5_K q and k beside a Q6_K v, as a Q5_K_M file has them."""
    from frink_amd import synth
    print("gemv group, mixed", flush=True)
    cols = 2048
    x = synth.activations(8, 1, cols)[0]
    kinds = [fo.Q5_K, fo.Q5_K, fo.Q6_K, fo.Q8_0, fo.Q8_0, fo.Q4_K, fo.Q5_K]
    data = [make_weights(k, 24 + i, cols, seed=70 + i) for i, k in enumerate(kinds)]
    ws = [fa.Weights.from_host(k, d, 24 + i, cols) for i, (k, d) in enumerate(zip(kinds, data))]
    for i, (k, d, y) in enumerate(zip(kinds, data, fa.gemv_multi(ws, to_dev(x)))):
        assert_rows_close(y.cpu().numpy()[None], fo.gemv(k, d, 24 + i, cols, x, fo.F32_DOT if k == fo.Q8_0 else fo.INT_DOT)[None], "mixed, matrix %d" % i)
    for w in ws:
        w.release()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [fo.Q5_K, fo.Q6_K, fo.Q8_0])
@pytest.mark.parametrize("blocks,ffn", [(2, 32), (4, 96), (5, 1568), (8, 2080), (9, 64), (15, 224), (16, 160), (17, 4128), (20, 32), (24, 2816), (28, 1120), (32, 96),
                                        (40, 672), (63, 64), (64, 3104), (66, 32)])
def test_gate_up_and_swiglu_in_one_launch(fa, kind, blocks, ffn):
    """frk_hip_ffn_swiglu_dev's gate and up against the two matrices' own GEMVs and the oracle's SwiGLU; the down projection is a
    Q8_0 diagonal, so that the result shows every intermediate (127 f16(1/127) times it, rounded twice)."""
    from frink_amd import synth
    print("glu", kind, blocks, ffn, flush=True)
    cols = 256 * blocks
    data = [make_weights(kind, ffn, cols, seed=11 * blocks + ffn + i) for i in range(2)]
    x = synth.activations(cols + ffn, 1, cols, outlier_frac=0.01)[0]
    scale = np.float16(1.0 / 127)
    diagonal = np.zeros((ffn, ffn // 32, 34), np.uint8)
    diagonal[:, :, :2] = np.frombuffer(scale.tobytes(), np.uint8)
    for i in range(ffn):
        diagonal[i, i // 32, 2 + i % 32] = 127
    wg, wu = (fa.Weights.from_host(kind, d, ffn, cols) for d in data)
    wd = fa.Weights.from_host(fo.Q8_0, diagonal.reshape(ffn, -1), ffn, ffn)
    got = fa.ffn_swiglu(wg, wu, wd, to_dev(x)).cpu().numpy()
    g, u = (w.gemv(to_dev(x)).cpu().numpy() for w in (wg, wu))
    want = fo.swiglu(g, u) * np.float32(127) * np.float32(scale)
    if kind == fo.Q5_K:  # (rows of 8 and 16 blocks alone: the whole-cache-line kernel, whose sums go in another order)
        assert_rows_close(got[None], want[None], "glu kind %d %dx%d" % (kind, ffn, cols))
    else:
        assert np.array_equal(bits(got), bits(want))
    for w in (wg, wu, wd):
        w.release()
