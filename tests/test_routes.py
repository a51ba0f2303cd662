"""Which kernels a call goes to, on the CPU (host_library.py): shapes that were timed on both of the kernels a rule chooses from, each
with the kernel that was the faster one, around the lines that the rules draw and beyond the sizes they were first fitted to."""
import pytest

import host_library
import oracle as fo

PROGRAM = r"""
#include <cstdio>
#include "frink_amd/csrc/frk_internal.hpp"
#include "include/frink_hip.h"
int main() {  // a call a line: its name, kind, rows, blocks of 256 columns, tokens; the kernels it launches
    char call[16];
    int kind;
    size_t rows, nb, batch;
    static float room[64];
    while (scanf("%15s %d %zu %zu %zu", call, &kind, &rows, &nb, &batch) == 5) {
        frk_weights w;
        w.kind = kind, w.rows = rows, w.cols = nb * 256, w.layout = frk::layout_for(kind, w.cols), w.dev = (uint8_t *)room;
        const std::string name = call;
        int rc = -99;
        if (name == "gemv") rc = frk_hip_gemv_dev(&w, room, room, FRK_ACT_F32, nullptr);
        if (name == "gemm") rc = frk_hip_gemm_dev(&w, room, batch, room, nullptr);
        if (name == "q8k") rc = frk_hip_gemm_q8k_dev(&w, (int8_t *)room, room, (int16_t *)room, batch, room, nullptr);
        printf("%d %s\n", rc, HipStub::get().take().c_str());
    }
}
"""


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    binary = host_library.build(tmp_path_factory.mktemp("routes"), PROGRAM)

    def of(calls):
        lines = host_library.run(binary, "".join("%s %d %d %d %d\n" % c for c in calls)).splitlines()
        assert len(lines) == len(calls)
        return [(int(line.split()[0]), line.split(None, 1)[1]) for line in lines]

    return of


def check(kernels, call, kind, shapes, kernel, taken):
    """shapes: (rows, blocks, tokens)"""
    got = kernels([(call, kind, r, nb, m) for r, nb, m in shapes])
    for shape, (rc, names) in zip(shapes, got):
        assert rc == 0, (shape, rc)
        assert (kernel in names) == taken, (call, kind, shape, names)


# us, a quantization launch and a GEMV / columns: 36784 x 12 blocks 22.0 / 21.3, 88059 x 12 39.0 / 41.9, 58054 x 15 31.3 / 33.7, 141333 x 9 55.3 / 46.0
def test_one_q5_k_row_of_9_to_15_blocks(kernels):
    check(kernels, "gemv", fo.Q5_K, [(512, 9, 1), (14336, 12, 1), (36784, 12, 1), (141333, 9, 1), (138618, 10, 1)], "gemv_q4_k_cols_kernel", True)
    check(kernels, "gemv", fo.Q5_K, [(88059, 12, 1), (58054, 15, 1), (68476, 12, 1)], "gemv_q4_k_cols_kernel", False)


# us, whole rows a wavefront / columns: Q4_K 4284 x 20 blocks 5.8 / 6.4, 4096 x 20 5.8 / 5.3, 6285 x 17 6.9 / 6.2; Q5_K 4439 x 20 6.9 / 7.7,
# 3948 x 20 6.6 / 6.5, 6285 x 17 10.9 / 9.1, 9980 x 21 12.8 / 13.2, 8192 x 21 12.4 / 11.5, 10128 x 22 17.3 / 13.5
def test_one_row_of_17_to_21_blocks(kernels):
    for kind, columns, rows in ((fo.Q4_K, [(512, 17), (4096, 20), (6285, 17), (8192, 20), (9980, 21)], [(4284, 20), (4710, 20), (5827, 19), (6144, 18), (8208, 20)]),
                                (fo.Q5_K, [(512, 17), (4096, 20), (6285, 17), (8192, 20), (2048, 21), (6285, 21), (8192, 21), (10128, 22), (16475, 23)],
                                 [(4439, 20), (5029, 19), (6144, 18), (8208, 20), (9980, 21), (12286, 21), (17631, 21)])):
        check(kernels, "gemv", kind, [s + (1,) for s in columns], "gemv_q4_k_cols_kernel", True)
        check(kernels, "gemv", kind, [s + (1,) for s in rows], "gemv_q4_k_cols_kernel", False)


# (us, what was there / sixteen-row workgroups; rows, blocks, tokens)
SIXTEEN_ROWS = {
    fo.Q4_K: [(4096, 16, 2), (4096, 43, 8), (14336, 16, 16), (4096, 56, 16), (4096, 16, 32), (5120, 56, 7), (12068, 44, 7), (17240, 31, 7), (7426, 64, 6), (16671, 38, 11), (135580, 16, 13),
              (7, 2, 32)],
    fo.Q5_K: [(4096, 43, 8), (4096, 43, 16), (4096, 16, 32), (9030, 49, 3), (7914, 125, 7), (33961, 31, 5), (3926, 92, 9), (16495, 18, 22), (154414, 4, 2)],
    fo.Q6_K: [(4096, 43, 8), (4096, 43, 32), (4096, 56, 32), (411, 127, 15), (421, 127, 27), (13840, 14, 23), (5537, 91, 10), (88582, 8, 8), (1376, 47, 19)],
}
OTHERS = {
    # thin kernels that fill a round: 22.3 / 24.1, 27.7 / 31.6, 43.8 / 59.0, 33.7 / 39.3, 73.1 / 92.3
    # their four tokens' form: 20.7 / 22.9; span: 8.9 / 9.5, 84.8 / 101
    # tiles: 19.2 / 20.2, 34.7 / 45.8, 18.5 / 24.3, 56.8 / 60.7, 54.2 / 62.4, 15.2 / 16.9
    fo.Q4_K: [(7659, 51, 6), (14336, 43, 6), (30394, 40, 6), (61849, 14, 7), (58326, 37, 5), (5961, 51, 3), (14336, 8, 5), (97913, 24, 15),
              (4193, 48, 13), (4689, 123, 16), (1322, 126, 11), (14889, 83, 12), (58128, 23, 10), (4956, 23, 17), (6785, 16, 2)],
    # 22.0 / 25.8, 28.9 / 31.9, 71.5 / 81.9; 38.8 / 47.3, 25.1 / 30.3, 26.3 / 38.5, 19.9 / 31.0
    fo.Q5_K: [(7432, 50, 3), (14755, 36, 7), (130371, 14, 3), (4532, 115, 10), (10256, 24, 27), (2108, 120, 21), (14559, 23, 19), (2084, 62, 24)],
    # 18.4 / 26.1, 19.8 / 32.1, 26.2 / 31.1, 27.5 / 30.0, 14.9 / 17.7, 13.8 / 15.0, 1.13 of the time
    fo.Q6_K: [(661, 117, 13), (921, 121, 18), (13840, 20, 22), (4233, 49, 28), (1064, 52, 23), (1069, 52, 11), (1024, 40, 28), (7398, 16, 2), (143833, 12, 8)],
}


@pytest.mark.parametrize("kind", [fo.Q4_K, fo.Q5_K, fo.Q6_K])
def test_two_to_thirty_two_tokens(kernels, kind):
    check(kernels, "gemm", kind, SIXTEEN_ROWS[kind], "gemm_k_rows_kernel", True)
    check(kernels, "gemm", kind, OTHERS[kind], "gemm_k_rows_kernel", False)


# (us, the pipelined GEMM / every 32 tokens by workgroups of their own)
SMALL = {fo.Q4_K: [(1101, 8, 103), (1115, 33, 90), (854, 32, 102), (369, 31, 295), (19, 2, 63)], fo.Q5_K: [(2146, 13, 70), (272, 71, 54), (385, 27, 298), (20, 2, 34)],
         fo.Q6_K: [(3856, 14, 52), (129, 75, 259), (63, 110, 33), (857, 42, 40), (18163, 3, 67)]}
# 18.5 / 21.3, 17.0 / 18.9, 17.6 / 19.0, 24.9 / 30.3, 12.3 / 15.4, 21.2 / 29.4; 22.3 / 24.8, 23.7 / 25.7, 35.5 / 39.1, 15.7 / 17.2; 11.7 / 13.3, 12.8 / 15.8, 22.3 / 29.2,
# 12.8 / 13.8, 1.18 of the time
LARGER = {fo.Q4_K: [(308, 29, 401), (2443, 31, 34), (1193, 27, 136), (144, 107, 63), (31622, 2, 63), (4704, 39, 53)], fo.Q5_K: [(2087, 43, 42), (1028, 27, 242), (42, 125, 115), (8551, 2, 248)],
          fo.Q6_K: [(284, 38, 34), (261, 52, 36), (3459, 22, 99), (12202, 2, 111), (3304, 6, 508)]}


@pytest.mark.parametrize("kind", [fo.Q4_K, fo.Q5_K, fo.Q6_K])
def test_more_tokens_of_small_matrices(kernels, kind):
    check(kernels, "gemm", kind, SMALL[kind], "gemm_k_rows_kernel", True)
    check(kernels, "gemm", kind, LARGER[kind], "gemm_k_rows_kernel", False)


# (us, the tiled form made first / plain rows, the same bits: 22.4 / 18.8, 13.4 / 10.4; 9.2 / 6.9, 15.5 / 12.2, 15.9 / 13.0; 11.3 / 8.7, 19.9 / 17.5)
PLAIN = {fo.Q4_K: [(13455, 26, 5), (5525, 24, 8)], fo.Q5_K: [(3945, 18, 8), (6956, 24, 8), (7518, 23, 14)], fo.Q6_K: [(6368, 12, 10), (14336, 16, 12)]}


@pytest.mark.parametrize("kind", [fo.Q4_K, fo.Q5_K, fo.Q6_K])
def test_a_batch_quantized_before_needs_no_tiles(kernels, kind):
    check(kernels, "q8k", kind, PLAIN[kind], "gemm_k_rows_kernel<%d,1,true>" % kind, True)
    check(kernels, "q8k", kind, PLAIN[kind], "tile_q8_k_kernel", False)
