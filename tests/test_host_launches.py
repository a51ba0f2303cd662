"""The decode launchers' host code under the address sanitizer, on the CPU: every kind, length and number of matrices that the
grouped launches take, each with an array of outputs no longer than it has matrices.  The HIP runtime is a stub that counts launches
(nothing reaches a device; the kernels' code is not compiled)."""
import os
import subprocess

from frink_amd import build as fb

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = r"""
#include <cstdio>
#include <vector>
#include "frink_amd/csrc/frk_internal.hpp"
static int launches;
extern "C" {
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *lds, hipStream_t *s) { *g = *b = dim3(1), *lds = 0, *s = nullptr; return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { launches++; return hipSuccess; }
hipError_t hipFuncSetAttribute(const void *, hipFuncAttribute, int) { return hipSuccess; }
hipError_t hipGetDevice(int *dev) { *dev = 0; return hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { *v = 256; return hipSuccess; }
hipError_t hipGetLastError() { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
void **__hipRegisterFatBinary(const void *) { static void *handle; return &handle; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
void __hipUnregisterFatBinary(void **) {}
}
namespace frk {
int set_error(int code, const char *, ...) { return code; }
}
using namespace frk;
static int failed, calls;
static void took(int rc, const char *what, size_t nb, size_t rows, size_t n) {
    calls++;
    if (rc != FRK_OK || launches != 1) printf("%s: %zu blocks, %zu rows, %zu matrices: status %d, %d launches\n", what, nb, rows, n, rc, launches), failed = 1;
    launches = 0;
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
    # (unoptimized: a read past a parameter is otherwise undefined before the sanitizer sees it)
    flags = ["-x", "hip", "--offload-arch=gfx950", "--offload-host-only", "-O0", "-g1", "-std=c++17", "-w", "-I", ROOT, "-Xarch_host", "-fsanitize=address"]
    (tmp_path / "launches.cpp").write_text(SOURCE)
    objs = []
    for src in (str(tmp_path / "launches.cpp"), os.path.join(fb.CSRC, "frk_gemv_direct.hip"), os.path.join(fb.CSRC, "frk_gemv_fused.hip")):
        objs.append(str(tmp_path / (os.path.basename(src) + ".o")))
        subprocess.check_call([fb.hipcc()] + flags + ["-c", src, "-o", objs[-1]])
    clang = "/opt/rocm/llvm/bin/clang++"
    binary = str(tmp_path / "launches")
    # (the kernels' image has no symbol in a host-only object)
    subprocess.check_call([clang, "-fsanitize=address", "-no-pie", "-Wl,--unresolved-symbols=ignore-all"] + objs + ["-o", binary])
    run = subprocess.run([binary], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, (run.stdout + run.stderr)[-3000:]
