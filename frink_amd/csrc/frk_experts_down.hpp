// The down projection of a mixture-of-experts layer for a token or a few, with the weighted sum of the token's experts
// (run_expert and combine_expert_outputs, crates/frink-moe/src/lib.rs:1068-1165 and 1246-1263):
//   out[token][row] = sum over the slots, in routing order, of  weight * (rows of expert ids[slot]) . act[token][slot]
// A workgroup takes a token's rows r .. r + rows_wg - 1 of ALL its slots, a wavefront a slot (slots w, w + 8, ... past
// eight): it quantizes the slot's intermediate to Q8_K for itself (bit-exact with quantize_activations_q8_k) while its
// weights are on their way, so nothing is shared before the sums, which meet in LDS behind the one barrier and are added
// there in the reference's order, each term a separate multiply and add.  With the sum in a launch of its own the pairs'
// rows went through memory and the layer paid a launch for them: 128 experts top-8 of 2048 / 768, one token, Q6_K, 5.6 + 3.0
// us under the profiler against 6.3 for this kernel.
// A launch of this size is bound by its latency (ids -> weights -> sums), not by its bytes (10 MB: 2 us).
#pragma once

#include "frk_device.hpp"

namespace frk {

// nb <= XB blocks a row; a row's units are shared by LPR lanes, and a wavefront has 64 / LPR * STEPS rows in flight.
// Unit: a lane's part of a row -- load(matrix, the row's offset, layout, unit), Act::load(quants, sums, scales, unit), dot(act).
constexpr int EXPERTS_DOWN_WAVES = 8, EXPERTS_DOWN_MAX_SLOTS = 64, EXPERTS_DOWN_ROWS = 8, EXPERTS_DOWN_MAX_ROWS = 64;
static __host__ __device__ inline size_t experts_down_act_bytes(int nb) { return (size_t)nb * (256 + 32 + 16); }

// SIMD_WAVES: wavefronts whose registers a SIMD holds.
template <class Unit, int LPR, int STEPS, int XB, int SIMD_WAVES>
__global__ __launch_bounds__(64 * EXPERTS_DOWN_WAVES, SIMD_WAVES) void experts_down_kernel(const uint8_t *__restrict__ W, Layout lay, int rows_e,
                                                                               int rows_wg, int nb, int n_experts, int k,
                                                                               const int32_t *__restrict__ ids,
                                                                               const float *__restrict__ weights,
                                                                               const float *__restrict__ act, float *__restrict__ out) {
    constexpr int PARTS = 64 / LPR, ROWS = PARTS * STEPS;
    static_assert(ROWS == EXPERTS_DOWN_ROWS, "rows a wavefront has in flight");
    extern __shared__ uint4 smem_down[];
    __shared__ float slot_weight[EXPERTS_DOWN_MAX_SLOTS];
    __shared__ int slot_id[EXPERTS_DOWN_MAX_SLOTS];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), waves = (int)blockDim.x >> 6;
    const int part = lane / LPR, l = lane % LPR;
    const size_t first = (size_t)blockIdx.y * k;
    const int row_begin = (int)blockIdx.x * rows_wg, row_end = min(rows_e, row_begin + rows_wg);
    const int units = nb * Unit::PER_BLOCK, u = min(l, units - 1);  // (a lane past the row's units repeats the last, unused)
    int8_t *const sq = reinterpret_cast<int8_t *>(smem_down) + (size_t)wave * experts_down_act_bytes(nb);
    int16_t *const sbs = reinterpret_cast<int16_t *>(sq + (size_t)nb * QK_K);
    float *const sd = reinterpret_cast<float *>(sbs + (size_t)nb * 16);
    float *const sums = reinterpret_cast<float *>(reinterpret_cast<int8_t *>(smem_down) + (size_t)waves * experts_down_act_bytes(nb));
    const bool lists = (int)threadIdx.x < k;
    const int list_id = lists ? ids[first + threadIdx.x] : 0;
    const float list_weight = lists ? weights[first + threadIdx.x] : 0.0f;

    for (int slot = wave; slot < k; slot += waves) {
        const int id = __builtin_amdgcn_readfirstlane(ids[first + slot]);
        const float *xs = act + (first + slot) * (size_t)nb * QK_K;
        float4 xv[XB];
#pragma unroll
        for (int b = 0; b < XB; b++) xv[b] = reinterpret_cast<const float4 *>(xs + (size_t)min(b, nb - 1) * QK_K)[lane];
        // (an id outside the experts computes on expert 0 and is left out of the sum)
        const uint8_t *We = W + (size_t)(id >= 0 && id < n_experts ? id : 0) * rows_e * lay.row_stride;
        Unit w[STEPS];
        auto request = [&](int r0) {
#pragma unroll
            for (int st = 0; st < STEPS; st++) w[st].load(We, (uint32_t)min(r0 + st * PARTS + part, rows_e - 1) * (uint32_t)lay.row_stride, lay, u);
        };
        request(row_begin);
        __builtin_amdgcn_sched_barrier(0);  // (every request is out before anything waits for the first of them)
#pragma unroll
        for (int b = 0; b < XB; b++) {
            float d;
            int s16;
            const uint32_t packed = quantize_q8_k_lane<false>(xv[b], d, s16);
            if (b < nb) {  // uniform
                reinterpret_cast<uint32_t *>(sq + b * QK_K)[lane] = packed;
                if ((lane & 3) == 0) sbs[b * 16 + (lane >> 2)] = (int16_t)s16;
                if (lane == 0) sd[b] = d;
            }
        }
        // (the wavefront's own LDS: read in order behind the writes, no barrier)
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        typename Unit::Act a;
        a.load(sq, sbs, sd, u);
        for (int r0 = row_begin; r0 < row_end; r0 += ROWS) {
            if (r0 != row_begin) request(r0);
#pragma unroll
            for (int st = 0; st < STEPS; st++) {
                const float v = part_sum<LPR>(l < units ? w[st].dot(a) : 0.0f);
                const int r = r0 + st * PARTS + part;
                if (l == 0 && r < row_end) sums[slot * rows_wg + r - row_begin] = v;
            }
        }
    }
    if (lists) {
        slot_id[threadIdx.x] = list_id;
        slot_weight[threadIdx.x] = list_weight;
    }
    __syncthreads();
    const int r = row_begin + (int)threadIdx.x;
    if ((int)threadIdx.x < rows_wg && r < row_end) {
        float acc = 0.0f;
        for (int s = 0; s < k; s++) {
            const int id = slot_id[s];
            if (id >= 0 && id < n_experts) acc += slot_weight[s] * sums[s * rows_wg + threadIdx.x];
        }
        out[(size_t)blockIdx.y * rows_e + r] = acc;
    }
}

int experts_down_rows_wg(size_t rows_e, size_t batch, int waves, int simd_waves);  // frk_gemv_direct.hip
static_assert(EXPERTS_DOWN_ROWS * 8 == EXPERTS_DOWN_MAX_ROWS && EXPERTS_DOWN_MAX_ROWS <= 64, "a thread a row, one wavefront at least");

template <class Unit, int LPR, int STEPS, int XB, int SIMD_WAVES>
static int launch_experts_down_as(const frk_weights *w, int n_experts, size_t rows_e, const float *act, const int32_t *ids,
                                  const float *weights, size_t batch, int k, float *out, hipStream_t s) {
    const int nb = (int)(w->cols / QK_K), waves = k < EXPERTS_DOWN_WAVES ? k : EXPERTS_DOWN_WAVES;
    const int rows_wg = experts_down_rows_wg(rows_e, batch, waves, SIMD_WAVES);
    const size_t lds = (size_t)waves * experts_down_act_bytes(nb) + (size_t)k * rows_wg * 4;
    hipLaunchKernelGGL((experts_down_kernel<Unit, LPR, STEPS, XB, SIMD_WAVES>), dim3((unsigned)((rows_e + rows_wg - 1) / rows_wg), (unsigned)batch),
                       dim3(64 * waves), lds, s, w->dev, w->layout, (int)rows_e, rows_wg, nb, n_experts, k, ids, weights, act, out);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(FRK_ERR_HIP, "experts_down launch: %s", hipGetErrorString(e));
    return FRK_OK;
}

}  // namespace frk
