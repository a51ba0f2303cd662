// Batched GEMM for Q6_K weights on the int8 matrix cores:  y[M][rows] = Q8_K(x)[M][cols] . W^T, the pipelined kernel of
// frk_gemm_pipe.hpp over the resident planar rows (ql | qh | sc | d, see layout_for).
// The arithmetic is gemm_q6_k_q8_row / dot_q6_k_q8 (crates/frink-quant/src/lib.rs:1033-1110): per 256-wide block the
// exact integer  isum = sum_g sc_g * sum_{i in g} (q6_i - 32) * a_i  over the sixteen 16-weight groups g, then
// acc += (d * da) * isum.  A lane's 16 bytes of a 32x32x32 operand are 16 consecutive weights of one row, i.e. exactly one
// group: the group's scale is a lane value.
#include "frk_gemm_pipe.hpp"

namespace frk {

template <int RG, int KS, int MT>
__global__ __launch_bounds__(512) void gemm_q6_k_pipe_kernel(GemmArgs g) {
    pipe_gemm<FRK_KIND_Q6_K, RG, KS, MT>(g);
}

// 64 rows x 32 tokens, for batches of up to 32 rows
__global__ __launch_bounds__(512) void batch_q6_k_pipe_kernel(GemmArgs g) { pipe_gemm<FRK_KIND_Q6_K, 2, 4, 1>(g); }

// y = the parts' sums added in the order of the parts: the same bits on every run
__global__ __launch_bounds__(256) void sum_parts_kernel(const float *__restrict__ partial, int parts, size_t n,
                                                        float *__restrict__ y) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    float acc = partial[i];
    for (int p = 1; p < parts; p++) acc += partial[(size_t)p * n + i];
    y[i] = acc;
}

int launch_sum_parts(const float *partial, int parts, size_t n, float *y, hipStream_t s) {
    hipLaunchKernelGGL(sum_parts_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, partial, parts, n, y);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(FRK_ERR_HIP, "launch of the sum of a split GEMM's parts: %s", hipGetErrorString(e));
    return FRK_OK;
}

int launch_pipe_q6_k(const GemmArgs &g, int rows_wg, hipStream_t s) {
    return rows_wg == 256   ? launch_pipe<FRK_KIND_Q6_K, 8, 1, 4>(gemm_q6_k_pipe_kernel<8, 1, 4>, g, s)
           : rows_wg == 128 ? launch_pipe<FRK_KIND_Q6_K, 4, 2, 2>(gemm_q6_k_pipe_kernel<4, 2, 2>, g, s)
                            : launch_pipe<FRK_KIND_Q6_K, 2, 4, 1>(batch_q6_k_pipe_kernel, g, s);
}

}  // namespace frk
