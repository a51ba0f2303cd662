"""The router at the edges of its register counts."""
import numpy as np
import pytest

import oracle as fo
from test_gpu_parity import fa, to_dev  # noqa: F401 (fa: the module's fixture)


@pytest.mark.gpu
@pytest.mark.parametrize("n_experts", [1, 2, 63, 64, 65, 128, 129, 256, 257, 511, 512, 513, 1000, 1024])
def test_router_at_the_edges_of_its_registers(fa, n_experts):
    """The oracle's weights bit for bit and its ids, ties to the lowest index, whatever the number of registers a lane."""
    rng = np.random.default_rng(n_experts)
    logits = rng.standard_normal((5, n_experts)).astype(np.float32)
    logits[1] = 0.5                                        # every probability the same
    logits[2, rng.integers(0, n_experts, 3)] = 9.0         # ties at the top
    logits[3] *= 60.0                                      # most exponentials vanish
    logits[4, : n_experts // 2] = -np.inf
    k = min(n_experts, 8)
    for norm in (False, True):
        ids, w = fa.route_top_k_softmax(to_dev(logits), k, norm)
        for r in range(5):
            want_ids, want_w = fo.route_top_k_softmax(logits[r], k, norm)
            assert np.array_equal(ids[r].cpu().numpy(), want_ids), (r, norm)
            assert np.array_equal(w[r].cpu().numpy().view(np.uint32), np.asarray(want_w, np.float32).view(np.uint32)), (r, norm)
