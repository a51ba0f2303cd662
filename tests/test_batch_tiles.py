"""The pipelined K-quant GEMM where its tiles are not filled.  Batches of 9 to 32 rows at the sizes of the 64 x 32 tiles: rows past the
last whole tile, blocks that do not divide by a step's four shares, parts of few blocks (most of them are gemm_k_rows_kernel's by
now; sizes that still go to the tiles are in test_thin_kernels.py).  Larger ones whose last token tile has few rows in use."""
import ctypes as C

import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import fa, make_weights, to_dev  # noqa: F401 (fa: the module's fixture)


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", [
    (fo.Q4_K, 64, 256, 17), (fo.Q4_K, 65, 512, 32), (fo.Q4_K, 127, 1280, 31), (fo.Q4_K, 1000, 7680, 9), (fo.Q4_K, 4160, 2304, 20),
    (fo.Q4_K, 33, 14336, 16), (fo.Q5_K, 64, 2560, 17), (fo.Q5_K, 70, 8192, 9), (fo.Q5_K, 300, 2816, 32), (fo.Q5_K, 8200, 2304, 33),
    (fo.Q5_K, 4700, 6144, 10), (fo.Q6_K, 1300, 6912, 17), (fo.Q6_K, 2400, 11008, 13), (fo.Q6_K, 2700, 7936, 32), (fo.Q6_K, 4200, 4352, 25),
    (fo.Q6_K, 4161, 12288, 9), (fo.Q6_K, 700, 7936, 33),
])
def test_batches_match_exact_arithmetic(fa, kind, rows, cols, batch):
    _check(fa, kind, rows, cols, batch)


def _check(fa, kind, rows, cols, batch):
    from bench import random_blocks
    from frink_amd import synth
    print("batch tiles", kind, rows, cols, batch, flush=True)
    data = random_blocks(kind, rows, cols, seed=rows + cols)
    x = synth.activations(batch, batch, cols, outlier_frac=0.01)
    w = fa.Weights.from_host(kind, data, rows, cols)
    got = w.gemm(to_dev(x)).cpu().numpy().astype(np.float64)
    w.release()
    a = np.empty((batch, cols), np.float64)
    for r in range(batch):
        q, d, _ = fo.quantize_q8_k(x[r])
        a[r] = (q.reshape(-1, 256).astype(np.float64) * d.astype(np.float64)[:, None]).ravel()
    wd = fo.dequant(kind, data).reshape(rows, cols).astype(np.float64)
    # Integers are exact up to the float step: a handful of f32 roundings a block (sum, scale, mins) of terms no larger than
    # the block's sum of magnitudes, one for each addition onto the running sum, one a share and one a part.  The dequantized
    # weights round twice an element.  (Mins: the two terms of a block cancel, each is bounded by |a| times the offsets.)
    mag = np.abs(a) @ np.abs(wd).T
    if kind != fo.Q6_K:
        mag = mag + np.abs(a).sum(1)[:, None] * np.abs(wd).max(1)[None, :]
    room = (cols // 256 + 24) * 2.0 ** -24 * mag
    assert (np.abs(got - a @ wd.T) <= room).all(), float((np.abs(got - a @ wd.T) / room).max())


@pytest.mark.gpu
@pytest.mark.parametrize("kind,rows,cols,batch", [
    (fo.Q4_K, 3000, 8192, 65), (fo.Q5_K, 2000, 8192, 97), (fo.Q6_K, 1024, 11008, 96), (fo.Q4_K, 2600, 8192, 129), (fo.Q5_K, 11008, 4096, 197),
    (fo.Q6_K, 11000, 4096, 170), (fo.Q4_K, 5000, 4352, 161), (fo.Q5_K, 8200, 2048, 225), (fo.Q6_K, 2900, 8192, 290), (fo.Q4_K, 3300, 6400, 321),
])
def test_last_token_tile_with_fewer_rows_in_use(fa, kind, rows, cols, batch):
    """One to three 32-token tiles of the last 128 in use, with and without parts of its own number."""
    _check(fa, kind, rows, cols, batch)


class _Plan(C.Structure):
    _fields_ = [("rows_wg", C.c_int), ("tok_wg", C.c_int), ("k_split", C.c_int), ("k_last", C.c_int)]


def _plan(kind, rows, batch, cols):
    import frink_amd
    f = frink_amd.lib()._ZN3frk9pipe_planEimmm  # frk::pipe_plan
    f.restype, f.argtypes = _Plan, [C.c_int, C.c_size_t, C.c_size_t, C.c_size_t]
    return f(kind, rows, batch, cols // 256)


# shapes whose last token tile has one to three 32-token tiles in use; at a full price for it they take the small tile
APART = [(fo.Q4_K, 5596, 68, 5632), (fo.Q4_K, 10897, 151, 2560), (fo.Q4_K, 14336, 96, 8192), (fo.Q5_K, 5816, 70, 4352), (fo.Q5_K, 5702, 144, 3840)]


@pytest.mark.parametrize("kind,rows,batch,cols", APART)
def test_a_partly_used_large_tile_takes_no_batch_from_the_small_one(kind, rows, batch, cols):
    """The large tile folds the mins into the sums, with two roundings a block more than the small one's."""
    assert _plan(kind, rows, batch, cols).rows_wg == 128


@pytest.mark.parametrize("kind,rows,batch,cols,sums", [
    (fo.Q6_K, 11516, 274, 12544, 3), (fo.Q6_K, 7777, 164, 8704, 4), (fo.Q5_K, 7196, 139, 5120, 4), (fo.Q5_K, 11008, 197, 4096, 2),
])
def test_no_token_tile_is_added_up_in_fewer_sums_than_at_a_full_price(kind, rows, batch, cols, sums):
    p = _plan(kind, rows, batch, cols)
    assert min(p.k_split, p.k_last) * (2 if p.rows_wg == 128 else 1) >= sums


def _block_terms(data, rows, cols, x):
    """(A, D, N, s1, s2) of every block: what the float step adds is A * (D * s1 + N * s2), s1 and s2 exact."""
    f = np.float32
    nb = cols // 256
    blk = data.reshape(rows, nb, 144)
    d = blk[:, :, 0:2].copy().view(np.float16)[:, :, 0].astype(f)
    dmin = blk[:, :, 2:4].copy().view(np.float16)[:, :, 0].astype(f)
    s = blk[:, :, 4:16].astype(np.int64)
    sc = np.concatenate((s[..., :4] & 63, (s[..., 8:] & 15) | (s[..., :4] >> 6 << 4)), -1)
    m = np.concatenate((s[..., 4:8] & 63, (s[..., 8:] >> 4) | (s[..., 4:8] >> 6 << 4)), -1)
    nib = blk[:, :, 16:].reshape(rows, nb, 4, 32)
    q = np.stack((nib & 15, nib >> 4), 3).reshape(rows, nb, 8, 32)
    aq, da = zip(*[fo.quantize_q8_k(r)[:2] for r in x])
    aq = np.stack(aq).reshape(len(x), nb, 8, 32).astype(np.float64)
    da = np.stack(da).reshape(len(x), nb).astype(f)
    terms = []
    for b in range(nb):
        s1 = aq[:, b].reshape(len(x), 256) @ (q[:, b] * sc[:, b, :, None]).reshape(rows, 256).astype(np.float64).T
        s2 = aq[:, b].sum(2) @ m[:, b].astype(np.float64).T
        terms.append(tuple(np.broadcast_to(v, s1.shape) for v in (da[:, b, None], d[:, b], -dmin[:, b])) + (s1, s2))
    return terms


def _fma(a, b, c):
    return (a.astype(np.float64) * b.astype(np.float64) + c.astype(np.float64)).astype(np.float32)


def _two_norm_errors(data, rows, cols, x, parts):
    """The 2-norm errors against 64-bit sums of the float step with a block's mins apart and folded, a row's blocks in so
    many sums added up in order: every operation of the kernel's float step in f32, in numpy."""
    f, fma = np.float32, _fma
    nb = cols // 256
    terms = _block_terms(data, rows, cols, x)
    exact, sums = 0.0, {"apart": [], "folded": []}
    for p in range(parts):
        acc = {k: np.zeros((len(x), rows), f) for k in sums}
        for b in range(nb * p // parts, nb * (p + 1) // parts):
            A, D, N, s1, s2 = terms[b]
            exact = exact + A.astype(np.float64) * (D.astype(np.float64) * s1 + N.astype(np.float64) * s2)
            acc["apart"] = fma(A, fma(N, s2.astype(f), D * s1.astype(f)), acc["apart"])
            c = ((D * (f(1) / N)) * s1.astype(f) + s2).astype(f)
            acc["folded"] = fma(A * N, c, acc["folded"])
        for k in sums:
            sums[k] = acc[k] if p == 0 else sums[k] + acc[k]
    return exact, {k: np.linalg.norm(v - exact) / np.linalg.norm(exact) for k, v in sums.items()}


@pytest.mark.gpu
@pytest.mark.parametrize("rows,batch,cols,parts", [APART[0][1:] + (4,), APART[1][1:] + (2,)])  # (two shares of two parts, of one)
def test_batches_of_the_small_tile_are_as_exact_as_its_float_step(fa, rows, batch, cols, parts):
    """The 2-norm error lies with the mins apart, not folded: below the middle of what the two float steps have."""
    from bench import random_blocks
    from frink_amd import synth
    print("small tile's error", rows, cols, batch, flush=True)
    data = random_blocks(fo.Q4_K, rows, cols, seed=rows)
    x = synth.activations(batch, batch, cols)
    w = fa.Weights.from_host(fo.Q4_K, data, rows, cols)
    got = w.gemm(to_dev(x)).cpu().numpy()[:, :64].astype(np.float64)
    w.release()
    exact, want = _two_norm_errors(data.reshape(rows, -1)[:64], 64, cols, x, parts)
    error = np.linalg.norm(got - exact) / np.linalg.norm(exact)
    print(error, want, flush=True)
    assert want["apart"] < 0.9 * want["folded"]
    assert error < (want["apart"] * want["folded"]) ** 0.5


def _in_pairs(v):
    while len(v) > 1:
        v = [v[i] + v[i + 1] if i + 1 < len(v) else v[i] for i in range(0, len(v), 2)]
    return v[0]


@pytest.mark.gpu
@pytest.mark.parametrize("rows,batch,cols", [(1304, 26, 11008), (1111, 28, 11520)])
def test_twelve_parts_are_added_in_pairs(fa, rows, batch, cols):
    """Twelve parts of a row, four shares each: below the middle of the 2-norm errors that adding them in order and in pairs have."""
    from bench import random_blocks
    from frink_amd import synth
    print("twelve parts' error", rows, cols, batch, flush=True)
    p = _plan(fo.Q4_K, rows, batch, cols)
    assert (p.rows_wg, p.k_split) == (64, 12)
    data = random_blocks(fo.Q4_K, rows, cols, seed=rows)
    x = synth.activations(batch, batch, cols)
    w = fa.Weights.from_host(fo.Q4_K, data, rows, cols)
    got = w.gemm(to_dev(x)).cpu().numpy()[:, :256].astype(np.float64)
    w.release()
    nb = cols // 256
    terms = _block_terms(data.reshape(rows, -1)[:256], 256, cols, x)
    exact = sum(A.astype(np.float64) * (D.astype(np.float64) * s1 + N.astype(np.float64) * s2) for A, D, N, s1, s2 in terms)
    parts = []
    for i in range(12):
        b0, b1 = nb * i // 12, nb * (i + 1) // 12
        steps = -(-(b1 - b0) // 4)
        shares = [np.zeros(exact.shape, np.float32) for _ in range(4)]
        for b in range(b0, b1):
            A, D, N, s1, s2 = terms[b]
            k = (b - b0) // steps
            shares[k] = _fma(A, _fma(N, s2.astype(np.float32), D * s1.astype(np.float32)), shares[k])
        parts.append(shares)
    order = sum(parts[0][1:], parts[0][0])
    for s in parts[1:]:
        order = order + sum(s[1:], s[0])
    want = {"order": order, "pairs": _in_pairs([_in_pairs(s) for s in parts])}
    assert all(v.dtype == np.float32 for v in want.values())
    want = {k: np.linalg.norm(v - exact) / np.linalg.norm(exact) for k, v in want.items()}
    error = np.linalg.norm(got - exact) / np.linalg.norm(exact)
    print(error, want, flush=True)
    assert want["pairs"] < 0.92 * want["order"]
    assert error < (want["pairs"] * want["order"]) ** 0.5


@pytest.mark.gpu
@pytest.mark.parametrize("rows,cols,batch", [(1264, 2048, 19), (300, 2048, 32), (4096, 3072, 23)])
def test_short_rows_stay_on_the_thin_kernels(fa, rows, cols, batch):
    """Q4_K of 8 and 12 blocks: a row's results do not depend on the batch that it came in with, up to 32 rows (on gemm_k_rows_kernel,
    as on the thin kernels before)."""
    from frink_amd import synth
    w = fa.Weights.from_host(fo.Q4_K, make_weights(fo.Q4_K, rows, cols, seed=rows), rows, cols)
    x = to_dev(synth.activations(batch, batch, cols))
    y, first = w.gemm(x).cpu().numpy(), w.gemm(x[:16].contiguous()).cpu().numpy()
    assert np.array_equal(y[:16].view(np.uint32), first.view(np.uint32))
    q8k = w.gemm_q8k(fa.quantize_q8_k(x.reshape(-1)), batch).cpu().numpy()
    assert np.array_equal(q8k.view(np.uint32), y.view(np.uint32))
    w.release()
