"""The bucketing of a mixture-of-experts batch (moe_group): up to 4096 pairs whose bits fit one round of the bit matrix, and more;
few and many experts (runs of the rows' words of 1 to 31 words), experts nobody chose, ids outside the experts."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import fa, to_dev  # noqa: F401 (fa: the module's fixture)


@pytest.mark.gpu
@pytest.mark.parametrize("n_experts,k,batch", [(1, 1, 32), (2, 2, 2048), (3, 1, 4096), (3, 1, 4097), (60, 4, 1000), (128, 8, 512), (128, 8, 513),
                                               (600, 1, 850), (600, 1, 1000), (1000, 2, 200), (1024, 1, 512), (1024, 1, 513), (700, 3, 230)])
def test_pairs_keep_their_order_in_every_bucket(fa, n_experts, k, batch):
    """Position of every pair in the order experts ascending, pairs ascending (pos_of), -1 for an id outside the experts."""
    import torch
    print("bucketing", n_experts, k, batch, flush=True)
    rng = np.random.default_rng(n_experts + batch)
    ids = np.stack([rng.permutation(n_experts)[:k] for _ in range(batch)]).astype(np.int32)
    if n_experts > 2:
        ids[ids == 1] = 0                      # nobody chose expert 1
        ids[rng.integers(0, batch, 5), 0] = (-1, n_experts, n_experts + 7, -5, 2 ** 30)
    gen = np.random.default_rng(1)
    from bench import random_blocks
    data = random_blocks(fo.Q4_K, n_experts * 256, 256, seed=3)
    w = fa.Weights.from_host(fo.Q4_K, data, n_experts * 256, 256)
    x = gen.standard_normal((batch, 256)).astype(np.float32)
    fa.moe_ffn(w, w, w, n_experts, to_dev(x), to_dev(ids), torch.ones((batch, k), device="cuda"))
    pos = fa.moe_intermediates(batch, k, n_experts, 256, 256)[4].cpu().numpy().ravel()
    flat = ids.ravel()
    valid = (flat >= 0) & (flat < n_experts)
    want = np.full(flat.size, -1, np.int64)
    order = np.flatnonzero(valid)[np.argsort(flat[valid], kind="stable")]
    want[order] = np.arange(order.size)
    w.release()
    assert np.array_equal(pos, want)
