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

// y = the parts' sums: the same bits on every run.  V floats a thread; PARTS > 0: that many parts, all asked for together and
// added in pairs, 0: any number, one after the other.  (Twelve parts of one to four blocks one after the other are as inexact as one sum of
// all blocks: 2-norm against 64 bits of 1179 x 9216 in Q5_K at 18 tokens 9.1e-8, in pairs 8.0e-8; the 128 x 64 tile, six parts in order, had 7.7e-8.)
template <int V, int PARTS>
__global__ __launch_bounds__(256) void sum_parts_kernel(const float *__restrict__ partial, int parts, size_t n,
                                                        float *__restrict__ y) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (i >= n) return;
    vec acc;
    if constexpr (PARTS > 0) {
        vec v[PARTS];
#pragma unroll
        for (int p = 0; p < PARTS; p++) v[p] = *reinterpret_cast<const vec *>(partial + (size_t)p * n + i);
#pragma unroll
        for (int p = PARTS; p > 1; p = (p + 1) / 2) {
#pragma unroll
            for (int i = 0; i < p / 2; i++) v[i] = v[2 * i] + v[2 * i + 1];
            if (p % 2) v[p / 2] = v[p - 1];
        }
        acc = v[0];
    } else {
        acc = *reinterpret_cast<const vec *>(partial + i);
        for (int p = 1; p < parts; p++) acc += *reinterpret_cast<const vec *>(partial + (size_t)p * n + i);
    }
    *reinterpret_cast<vec *>(y + i) = acc;
}

// Sums begin .. end - 1 of n, parts0 parts of those in front of `split` and parts1 of the others
template <int V>
__global__ __launch_bounds__(256) void sum_parts_apart_kernel(const float *__restrict__ partial, size_t n, size_t begin, size_t end, size_t split,
                                                              int parts0, int parts1, float *__restrict__ y) {
    typedef float vec __attribute__((ext_vector_type(V)));
    const size_t i = begin + ((size_t)blockIdx.x * 256 + threadIdx.x) * V;
    if (i >= end) return;
    const int parts = i < split ? parts0 : parts1;
    vec acc = *reinterpret_cast<const vec *>(partial + i);
    for (int p0 = 1; p0 < parts; p0 += 4) {  // four asked for together
        vec v[4];
#pragma unroll
        for (int k = 0; k < 4; k++) v[k] = *reinterpret_cast<const vec *>(partial + (size_t)min(p0 + k, parts - 1) * n + i);
#pragma unroll
        for (int k = 0; k < 4; k++) acc = p0 + k < parts ? acc + v[k] : acc;
    }
    *reinterpret_cast<vec *>(y + i) = acc;
}
int launch_sum_parts_apart(const float *partial, size_t n, size_t begin, size_t end, size_t split, int parts0, int parts1, float *y, hipStream_t s) {
    if (end <= begin) return FRK_OK;
    const bool by_four = (n | begin | end | split) % 4 == 0 && ((reinterpret_cast<uintptr_t>(partial) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
    const size_t per_wg = by_four ? 1024 : 256;
    const dim3 grid((unsigned)((end - begin + per_wg - 1) / per_wg));
    if (by_four) hipLaunchKernelGGL(sum_parts_apart_kernel<4>, grid, dim3(256), 0, s, partial, n, begin, end, split, parts0, parts1, y);
    else hipLaunchKernelGGL(sum_parts_apart_kernel<1>, grid, dim3(256), 0, s, partial, n, begin, end, split, parts0, parts1, y);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(FRK_ERR_HIP, "launch of the sum of a split GEMM's parts: %s", hipGetErrorString(e));
    return FRK_OK;
}

template <int V>
static void go_sum_parts(const float *partial, int parts, size_t n, float *y, hipStream_t s) {
    const dim3 grid((unsigned)((n / V + 255) / 256));
#define FRK_GO(P) hipLaunchKernelGGL((sum_parts_kernel<V, P>), grid, dim3(256), 0, s, partial, parts, n, y)
    if (parts == 2) FRK_GO(2);
    else if (parts == 3) FRK_GO(3);
    else if (parts == 4) FRK_GO(4);
    else if (parts == 5) FRK_GO(5);
    else if (parts == 6) FRK_GO(6);
    else if (parts == 8) FRK_GO(8);
    else if (parts == 12) FRK_GO(12);
    else if (parts == 16) FRK_GO(16);
    else FRK_GO(0);
#undef FRK_GO
}
int launch_sum_parts(const float *partial, int parts, size_t n, float *y, hipStream_t s) {
    // (Four floats a thread where that still fills the chip: with all parts asked for together 512 x 4096 of four parts 8.4 -> 7.0 us
    // under the profiler, 197 x 11008 of two 6.1 -> 5.6; 13 x 4096 of four 0.15 us faster with one float a thread.  A sum in
    // the GEMM by the last part to arrive was slower: its stores, the counter and the loads behind it are one wavefront's
    // chain of trips to memory, 512 x 4096 x 14336 94.2 -> 100.4 us.)
    const bool by_four = n >= (size_t)1 << 18 && n % 4 == 0 && ((reinterpret_cast<uintptr_t>(partial) | reinterpret_cast<uintptr_t>(y)) & 15) == 0;
    if (by_four) go_sum_parts<4>(partial, parts, n, y, s);
    else go_sum_parts<1>(partial, parts, n, y, s);
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
