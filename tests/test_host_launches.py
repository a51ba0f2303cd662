"""The decode launchers' host code under the address sanitizer, on the CPU: every kind, length and number of matrices that the
grouped launches take, each with an array of outputs no longer than it has matrices."""
import host_library

PROGRAM = r"""
#include <cstdio>
#include "frink_amd/csrc/frk_internal.hpp"
using namespace frk;
static int failed, calls;
static void took(int rc, const char *what, size_t nb, size_t rows, size_t n) {
    calls++;
    const size_t launches = HipStub::get().launched.size();
    if (rc != FRK_OK || launches != 1) printf("%s: %zu blocks, %zu rows, %zu matrices: status %d, %zu launches\n", what, nb, rows, n, rc, launches), failed = 1;
    HipStub::get().launched.clear();
}
int main() {
    const int kinds[] = {FRK_KIND_Q4_K, FRK_KIND_Q5_K, FRK_KIND_Q6_K, FRK_KIND_Q8_0};
    std::vector<float> room(1 << 12);  // (addresses only: nothing runs)
    std::vector<uint8_t> bytes(1 << 12);
    for (int kind : kinds)
        for (size_t nb = 1; nb <= 64; nb++)
            for (size_t rows : {1, 40, 1024, 4864, 14336}) {
                for (size_t n = 1; n <= 4; n++) {
                    std::vector<frk_weights> w(n);
                    std::vector<const frk_weights *> ws(n);
                    std::vector<float *> ys(n);
                    for (size_t i = 0; i < n; i++) {
                        w[i].kind = kind, w[i].rows = i ? (rows + 3) / 4 : rows, w[i].cols = nb * 256;
                        w[i].layout = layout_for(kind, w[i].cols), w[i].dev = bytes.data();
                        ws[i] = &w[i], ys[i] = room.data();
                    }
                    if (kind == FRK_KIND_Q4_K && n > 1) took(launch_gemv_q4_k_group(ws.data(), n, room.data(), ys.data(), nullptr), "Q4_K", nb, rows, n);
                    if (kind == FRK_KIND_Q5_K) took(launch_gemv_q5_k_group(ws.data(), n, room.data(), ys.data(), nullptr), "Q5_K", nb, rows, n);
                    if (kind == FRK_KIND_Q6_K && (direct_gemv_fits(ws[0]) || q6_k_cols_form(ws[0])))
                        took(launch_gemv_q6_k_group(ws.data(), n, room.data(), ys.data(), nullptr), "Q6_K", nb, rows, n);
                    if (kind == FRK_KIND_Q8_0 && q8_0_cols_form(ws[0]))
                        took(launch_gemv_q8_0_f32_group(ws.data(), n, room.data(), ys.data(), nullptr), "Q8_0", nb, rows, n);
                }
                frk_weights gate, up;
                for (frk_weights *w : {&gate, &up})
                    w->kind = kind, w->rows = rows, w->cols = nb * 256, w->layout = layout_for(kind, w->cols), w->dev = bytes.data();
                float *const act = room.data();
                if (kind == FRK_KIND_Q4_K) took(launch_gemv_q4_k_glu(&gate, &up, room.data(), act, nullptr), "Q4_K pair", nb, rows, 2);
                if (kind == FRK_KIND_Q5_K) took(launch_gemv_q5_k_glu(&gate, &up, room.data(), act, nullptr), "Q5_K pair", nb, rows, 2);
                if (kind == FRK_KIND_Q6_K && q6_k_cols_form(&gate)) took(launch_gemv_q6_k_glu(&gate, &up, room.data(), act, nullptr), "Q6_K pair", nb, rows, 2);
                if (kind == FRK_KIND_Q8_0 && q8_0_cols_form(&gate)) took(launch_gemv_q8_0_f32_glu(&gate, &up, room.data(), act, nullptr), "Q8_0 pair", nb, rows, 2);
            }
    printf("%d calls\n", calls);
    return failed;
}
"""


def test_grouped_and_paired_launches_stay_inside_their_arrays(tmp_path):
    calls = int(host_library.run(host_library.build(tmp_path, PROGRAM)).split()[0])
    assert calls == 5 * (64 * 3 + 64 * 4 + 64 * 4 + 62 * 4 + 64 + 64 + 53 + 62)
