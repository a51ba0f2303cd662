"""The down projection of a mixture-of-experts layer with the weighted sum in its launch (frk_experts_down.hpp): one slot,
slots past eight, rows that are not a multiple of a workgroup's, one to nine blocks a row, both kinds."""
import pytest

import oracle as fo
from test_gpu_parity import _moe_case, fa  # noqa: F401 (fa: the module's fixture)


@pytest.mark.gpu
@pytest.mark.parametrize("down_kind", [fo.Q4_K, fo.Q6_K])
@pytest.mark.parametrize("n_experts,k,hidden,ffn,batch", [
    (4, 1, 256, 256, 1), (8, 3, 768, 1024, 2), (16, 9, 512, 1280, 3), (12, 12, 2048, 512, 16), (9, 7, 1280, 1536, 5),
    (4, 2, 3072, 1792, 7), (4, 4, 256, 2304, 2),
])
def test_down_projection_with_the_weighted_sum(fa, n_experts, k, hidden, ffn, batch, down_kind):
    print("experts down", down_kind, n_experts, k, hidden, ffn, batch, flush=True)
    _moe_case(fa, n_experts, k, hidden, ffn, batch, seed=n_experts + 31 * batch, down_kind=down_kind)
