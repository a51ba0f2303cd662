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
