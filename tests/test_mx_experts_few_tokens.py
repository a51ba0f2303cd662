"""A token or a few through MXFP4 experts (frk_mx_experts.hip): rows of one block and of 96, numbers of blocks around the
sixteen lanes of a row, slots past the eight wavefronts of a workgroup, rows of down that no workgroup's share divides, ids
outside the experts, blocks of zeros."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import _end_to_end_gate, _other_kind_blocks, fa, to_dev  # noqa: F401 (fa: the module's fixture)


@pytest.mark.gpu
@pytest.mark.parametrize("n_experts,k,hidden,ffn,batch", [
    (2, 1, 32, 32, 1), (4, 2, 512, 544, 3), (12, 11, 480, 1024, 2), (8, 4, 1056, 2176, 5), (3, 2, 3072, 96, 31), (4, 4, 2880, 3072, 1),
    (64, 64, 64, 64, 2),
])
def test_few_tokens_through_mxfp4_experts(fa, n_experts, k, hidden, ffn, batch):
    from frink_amd import synth
    print("mx experts", n_experts, k, hidden, ffn, batch, flush=True)
    data = [_other_kind_blocks(fo.MXFP4, n_experts * r, c, seed=51 + i) for i, (r, c) in enumerate(((ffn, hidden), (ffn, hidden), (hidden, ffn)))]
    for d in data:
        d.reshape(-1, 17)[:, 0] = 110 + d.reshape(-1, 17)[:, 0] % 12
    x = synth.activations(54, batch, hidden)
    x[0, 32:64] = 0.0
    rng = np.random.default_rng(55)
    ids = np.stack([rng.permutation(n_experts)[:k] for _ in range(batch)]).astype(np.int32)
    w = rng.uniform(0.1, 1.0, (batch, k)).astype(np.float32)
    if batch > 1:
        ids[1, 0], ids[batch - 1, k - 1] = -1, n_experts
    hs = [fa.Weights.from_host(fo.MXFP4, d, r, c) for d, (r, c) in zip(data, ((n_experts * ffn, hidden), (n_experts * ffn, hidden), (n_experts * hidden, ffn)))]
    got = fa.moe_ffn(hs[0], hs[1], hs[2], n_experts, to_dev(x), to_dev(ids), to_dev(w)).cpu().numpy()
    g, u, d = (m.reshape(n_experts, -1) for m in data)
    want = np.zeros((batch, hidden), np.float32)
    for t in range(batch):
        for s in range(k):
            e = ids[t, s]
            if 0 <= e < n_experts:
                a = fo.swiglu(fo.gemm(fo.MXFP4, g[e], ffn, hidden, x[t:t + 1], fo.INT_DOT).ravel(), fo.gemm(fo.MXFP4, u[e], ffn, hidden, x[t:t + 1], fo.INT_DOT).ravel())
                want[t] += w[t, s] * fo.gemm(fo.MXFP4, d[e], hidden, ffn, a.reshape(1, ffn), fo.INT_DOT)[0]
    _end_to_end_gate(got, want, "mx experts E=%d k=%d %d/%d batch=%d" % (n_experts, k, hidden, ffn, batch), False)
    for h in hs:
        h.release()
