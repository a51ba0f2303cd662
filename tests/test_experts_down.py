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


@pytest.mark.parametrize("rows_e,batch,waves,simd_waves,rows", [
    (2048, 15, 1, 3, 16), (2048, 1, 8, 4, 8), (3840, 13, 6, 4, 56), (512, 5, 6, 3, 16), (5120, 10, 8, 3, 56), (2048, 4, 4, 4, 16), (1, 1, 1, 5, 8), (1 << 20, 16, 8, 3, 64),
])
def test_rows_of_a_workgroup_by_how_many_fit_a_cu(rows_e, batch, waves, simd_waves, rows):
    import ctypes as C

    import frink_amd
    f = frink_amd.lib()._ZN3frk20experts_down_rows_wgEmmii  # frk::experts_down_rows_wg
    f.restype, f.argtypes = C.c_int, [C.c_size_t] * 2 + [C.c_int] * 2
    assert f(rows_e, batch, waves, simd_waves) == rows


@pytest.mark.parametrize("kind,rows,ffn,batch,k,takes", [
    (fo.Q6_K, 512, 1024, 1, 16, True), (fo.Q6_K, 2304, 256, 1, 48, False), (fo.Q4_K, 2304, 256, 16, 48, True), (fo.Q4_K, 512, 256, 1, 64, False),
    (fo.Q6_K, 2048, 1280, 16, 4, True), (fo.Q6_K, 2048, 1280, 7, 6, True), (fo.Q6_K, 2048, 1280, 8, 6, False), (fo.Q6_K, 2048, 1536, 16, 8, True),
    (fo.Q4_K, 2048, 1536, 16, 7, True), (fo.Q4_K, 2048, 1536, 1, 9, False), (fo.Q6_K, 5120, 2048, 1, 5, False), (fo.Q6_K, 2816, 1792, 1, 8, True), (fo.Q4_K, 2816, 1792, 1, 8, False), (fo.Q6_K, 2816, 1792, 1, 9, False),
    (fo.Q4_K, 512, 1792, 1, 9, False), (fo.Q4_K, 512, 2048, 1, 4, True), (fo.Q4_K, 512, 2304, 1, 1, False),
])
def test_where_the_sum_is_in_the_down_projection(kind, rows, ffn, batch, k, takes):
    import ctypes as C

    import frink_amd
    f = frink_amd.lib()._ZN3frk18experts_down_takesEimmmm  # frk::experts_down_takes
    f.restype, f.argtypes = C.c_bool, [C.c_int] + [C.c_size_t] * 4
    assert f(kind, rows, ffn, batch, k) == takes
