"""Infinities, NaN and values whose products overflow in the activations of gemm_k_rows_kernel and of the MXFP4 experts' few-token
kernels: what the oracle has, where it has it, and the other rows keep their bits."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import _other_kind_blocks, bits, fa, make_weights, to_dev  # noqa: F401 (fa: the module's fixture)

pytestmark = pytest.mark.gpu


def _same_kind(got, want):
    """NaN where the oracle has it, infinities of its sign but where a finite value is within rounding of one, the rest close."""
    edge = np.abs(want) > 3.4e38
    assert np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(np.isinf(got)[~edge], np.isinf(want)[~edge])
    inf = np.isinf(want) & np.isinf(got)
    assert np.array_equal(np.sign(got[inf]), np.sign(want[inf]))
    both = np.isfinite(got) & np.isfinite(want)
    scale = np.abs(np.where(both, want, 0.0)).max(axis=1, keepdims=True)
    assert (np.abs(np.where(both, got, 0.0) / np.maximum(scale, 1e-30) - np.where(both, want, 0.0) / np.maximum(scale, 1e-30)) <= 1e-3).all()


@pytest.mark.parametrize("kind,rows,cols,batch", [(fo.Q4_K, 37, 1280, 7), (fo.Q4_K, 20, 2304, 21), (fo.Q5_K, 33, 1280, 9), (fo.Q5_K, 17, 768, 40), (fo.Q6_K, 19, 1280, 8),
                                                  (fo.Q6_K, 35, 4352, 29)])
def test_k_quant_batches(fa, kind, rows, cols, batch):
    from frink_amd import synth
    print("non-finite rows", kind, rows, cols, batch, flush=True)
    w = fa.Weights.from_host(kind, make_weights(kind, rows, cols, seed=rows), rows, cols)
    data = make_weights(kind, rows, cols, seed=rows)
    x = synth.activations(batch, batch, cols)
    plain = w.gemm(to_dev(x)).cpu().numpy()
    x[1, 300] = np.inf                    # a scale of infinity over zeros
    x[2, [0, 255, cols - 1]] = np.nan     # (counts as zero)
    x[3, 256:512] *= np.float32(1e38) / np.abs(x[3, 256:512]).max()   # products past the largest float
    x[4, 0], x[4, 700] = -np.inf, 1e30
    x[batch - 1, :256] = np.nan           # a block of nothing
    with np.errstate(all="ignore"):
        want = fo.gemm(kind, data, rows, cols, x)
    for got in (w.gemm(to_dev(x)), w.gemm_acts(fa.BatchActs(batch, cols).quantize(to_dev(x)))) + (
            (w.gemm_q8k(fa.quantize_q8_k(to_dev(x.reshape(-1))), batch),) if batch <= 32 else ()):
        got = got.cpu().numpy()
        _same_kind(got, want)
        others = [r for r in range(batch) if r not in (1, 2, 3, 4, batch - 1)]
        assert np.array_equal(bits(got[others]), bits(plain[others]))
    assert np.isnan(want[1]).all() and np.isnan(want[4]).all() and np.isfinite(want[2]).all()
    w.release()


@pytest.mark.parametrize("hidden,ffn,batch", [(416, 448, 6), (1600, 1216, 5), (2400, 1984, 7)])  # (four and five, three and four blocks a lane)
def test_few_tokens_through_mxfp4_experts(fa, hidden, ffn, batch):
    print("non-finite tokens through mxfp4 experts", hidden, ffn, batch, flush=True)
    n_experts, k = 3, 2
    rng = np.random.default_rng(hidden)
    data = [_other_kind_blocks(fo.MXFP4, n_experts * r, c, seed=60 + i) for i, (r, c) in enumerate(((ffn, hidden), (ffn, hidden), (hidden, ffn)))]
    for d in data:
        d.reshape(-1, 17)[:, 0] = 118 + d.reshape(-1, 17)[:, 0] % 4
    x = rng.standard_normal((batch, hidden)).astype(np.float32)
    ids = np.stack([rng.permutation(n_experts)[:k] for _ in range(batch)]).astype(np.int32)
    wt = rng.uniform(0.2, 1.0, (batch, k)).astype(np.float32)
    hs = [fa.Weights.from_host(fo.MXFP4, d, n_experts * r, c) for d, (r, c) in zip(data, ((ffn, hidden), (ffn, hidden), (hidden, ffn)))]
    plain = fa.moe_ffn(*hs, n_experts, to_dev(x), to_dev(ids), to_dev(wt)).cpu().numpy()
    x[0, 40] = np.inf        # its block's scale is infinite, its quants zeros: NaN in every gate, and NaN counts as zero on the way down
    x[1, [3, 390]] = 2.0e7   # scales past f16: infinite gates and ups, and NaN of those
    x[2, [5, 64]] = np.nan   # (counts as zero)
    x[3, :32] = np.nan
    got = fa.moe_ffn(*hs, n_experts, to_dev(x), to_dev(ids), to_dev(wt)).cpu().numpy()
    g, u, d = (m.reshape(n_experts, -1) for m in data)
    want = np.zeros((batch, hidden), np.float32)
    with np.errstate(all="ignore"):
        for t in range(batch):
            for s in range(k):
                e = ids[t, s]
                a = fo.swiglu(*(fo.gemm(fo.MXFP4, m[e], ffn, hidden, x[t:t + 1], fo.INT_DOT).ravel() for m in (g, u)))
                want[t] += wt[t, s] * fo.gemm(fo.MXFP4, d[e], hidden, ffn, a.reshape(1, ffn), fo.INT_DOT)[0]
    assert not want[0].any() and np.isnan(want[1]).all() and np.isfinite(want[2:]).all()
    assert not got[0].any() and np.isnan(got[1]).all()
    # (an intermediate's last bit now and then moves a quant of the down projection's input to the next level)
    assert (np.abs(got[2:] - want[2:]).max(axis=1) <= 1e-2 * np.abs(want[2:]).max(axis=1)).all()
    assert np.array_equal(bits(got[4:]), bits(plain[4:]))
    for h in hs:
        h.release()
