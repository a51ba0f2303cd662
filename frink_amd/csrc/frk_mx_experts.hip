// A token or a few through MXFP4 experts: every (token, slot) pair reads its expert's three matrices alone (run_expert,
// crates/frink-moe/src/lib.rs:1068-1165), on the integer tier (dot_mxfp4_q8, crates/frink-quant/src/legacy_q8.rs:169-213),
// in two launches:
//   gate and up of 32 rows of a pair, the token's row quantized to Q8_0 by every workgroup for itself, and their
//     silu(gate) * up, one Q8_0 block of the down projection's input, quantized where it is made;
//   down of all of a token's pairs and their weighted sum, a wavefront a slot, as frk_experts_down.hpp does it.
// Sixteen lanes share a row, a lane has every sixteenth block of 32 weights: up to six 16-byte loads a row and their scale
// bytes, all in flight before anything is waited for.
//
// In their place were five launches -- the tokens quantized, a row a wavefront for gate and up, silu and quantization, a row a
// wavefront for down, the sum -- whose workgroups staged an activation row for eight weight rows each.
// What bounds them: a launch's chain of ids -> weights -> sums for a token or two, then the vector ALU, two instructions a
// weight (a code goes through two byte look-ups, its sign picks one).
#include "frk_device.hpp"

namespace frk {

constexpr int MXE_LANES = 16, MXE_PARTS = 64 / MXE_LANES;  // lanes of a row, rows of a wavefront at a time
constexpr int MXE_MAX_UNITS = 6 * MXE_LANES;
constexpr int MXE_MAX_SLOTS = 64, MXE_WAVES = 8, MXE_MAX_ROWS = 64;

#if defined(__HIP_DEVICE_COMPILE__)
struct MxeSigned {
    uint32_t low, high;  // of the low nibbles, of the high ones
};
// eight E2M1 codes as twice their values, signed bytes
__device__ __forceinline__ MxeSigned mxe_signed(uint32_t w) {
    const uint32_t low = w & 0x07070707u, high = (w >> 4) & 0x07070707u;
    auto positive = [](uint32_t sel) { return __builtin_amdgcn_perm(0x0C080604u, 0x03020100u, sel); };
    auto negative = [](uint32_t sel) { return __builtin_amdgcn_perm(0xF4F8FAFCu, 0xFDFEFF00u, sel); };
    // (selectors 8 .. 11: the signs of bytes 1, 3, 5 and 7 of the pair, eight times each)
    const uint32_t sign_high = __builtin_amdgcn_perm(w, w << 8, 0x0b090a08u), sign_low = __builtin_amdgcn_perm(w << 4, w << 12, 0x0b090a08u);
    return {(negative(low) & sign_low) | (positive(low) & ~sign_low), (negative(high) & sign_high) | (positive(high) & ~sign_high)};
}

// A lane's blocks of a row: l, l + 16, ... (past the row's end the last one, unused)
template <int S>
struct MxeRow {
    uint4 codes[S];
    uint32_t scale[S];
    __device__ __forceinline__ void load(const uint8_t *row, int l, int units) {
#pragma unroll
        for (int s = 0; s < S; s++) codes[s] = reinterpret_cast<const uint4 *>(row)[min(l + s * MXE_LANES, units - 1)];
#pragma unroll
        for (int s = 0; s < S; s++) scale[s] = row[units * 16 + min(l + s * MXE_LANES, units - 1)];
    }
    // block s times its quants a, b of scale d: one rounding, then the sums' (gemv_units_int_kernel's)
    __device__ __forceinline__ float term(int s, const uint4 &a, const uint4 &b, float d) const {
        const uint32_t w[4] = {codes[s].x, codes[s].y, codes[s].z, codes[s].w};
        const uint32_t av[4] = {a.x, a.y, a.z, a.w}, bv[4] = {b.x, b.y, b.z, b.w};
        int isum = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const MxeSigned c = mxe_signed(w[i]);
            isum = dot4(c.low, av[i], isum);
            isum = dot4(c.high, bv[i], isum);
        }
        const uint32_t e = scale[s];  // ggml_e8m0_to_fp32_half: 2^(e - 128), the two subnormal patterns for e < 2
        const float half = __uint_as_float(e < 2 ? 0x00200000u << e : (e - 1) << 23);
        return d * (half * (float)isum);
    }
};
// a lane's terms added in pairs, then the lanes' sums
template <int S>
__device__ __forceinline__ float mxe_sum(float (&t)[S]) {
#pragma unroll
    for (int n = S; n > 1; n = (n + 1) / 2) {
#pragma unroll
        for (int i = 0; i < n / 2; i++) t[i] = t[2 * i] + t[2 * i + 1];
        if (n % 2) t[n / 2] = t[n - 1];
    }
    return part_sum<MXE_LANES>(t[0]);
}
#endif

struct MxeGateUpArgs {
    const uint8_t *gate, *up;
    size_t row_stride;
    int ffn, units, n_experts, k;  // units: blocks of a row
    const int32_t *ids;
    const float *x;
    int8_t *q;  // [pair][ffn]
    float *d;   // [pair][ffn / 32]
};
template <int S>
__global__ __launch_bounds__(512, 4) void mx_experts_gate_up_kernel(MxeGateUpArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
    __shared__ uint4 sq[2 * MXE_MAX_UNITS];
    __shared__ __align__(16) float gates[32];  // (read as float4 too)
    __shared__ float sd[MXE_MAX_UNITS], ups[32];
    __shared__ uint64_t table[32];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, l = lane % MXE_LANES, part = lane / MXE_LANES;
    const int pair = blockIdx.y, id = g.ids[pair];
    if (id < 0 || id >= g.n_experts) return;  // (uniform; the pair's activations are not read either)
    const int units = g.units;
    const float4 *const xs = reinterpret_cast<const float4 *>(g.x + (size_t)(pair / g.k) * units * 32);
    float4 xv[2];  // eight lanes a block
#pragma unroll
    for (int i = 0; i < 2; i++) xv[i] = xs[min(tid + 512 * i, units * 8 - 1)];
    const size_t row = ((size_t)id * g.ffn + (size_t)blockIdx.x * 32 + wave * MXE_PARTS + part) * g.row_stride;
    MxeRow<S> gate, up;
    gate.load(g.gate + row, l, units);
    up.load(g.up + row, l, units);
    __builtin_amdgcn_sched_barrier(0);  // (every request is out before anything waits for the first of them)
    if (tid < 32) table[tid] = EXPF_TABLE[tid];
    auto quantize = [&](float4 v, uint32_t &q) {  // quantize_activations_q8, Avx form; the block's scale
        float amax = fmaxf(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))), 0.0f);
        amax = fmaxf(amax, dpp_f<DPP_QUAD_XOR1>(amax));
        amax = fmaxf(amax, dpp_f<DPP_QUAD_XOR2>(amax));
        amax = fmaxf(amax, dpp_f<DPP_HALF_MIRROR>(amax));
        const float inv = amax != 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
        q = quants_of(quant_of(v.x * inv), quant_of(v.y * inv), quant_of(v.z * inv), quant_of(v.w * inv));
        return h2f(f2h_bits(__fdiv_rn(amax, 127.0f)));
    };
#pragma unroll
    for (int i = 0; i < 2; i++) {
        const int t = tid + 512 * i;
        uint32_t q;
        const float d = quantize(xv[i], q);
        if (t < units * 8) {
            reinterpret_cast<uint32_t *>(sq)[t] = q;
            if ((t & 7) == 0) sd[t >> 3] = d;
        }
    }
    lds_barrier();
    float tg[S], tu[S];
#pragma unroll
    for (int s = 0; s < S; s++) {
        const int u = l + s * MXE_LANES, at = min(u, units - 1);
        const uint4 a = sq[2 * at], b = sq[2 * at + 1];
        const float d = sd[at];
        tg[s] = u < units ? gate.term(s, a, b, d) : 0.0f;
        tu[s] = u < units ? up.term(s, a, b, d) : 0.0f;
    }
    const float vg = mxe_sum(tg), vu = mxe_sum(tu);
    if (l == 0) gates[wave * MXE_PARTS + part] = vg, ups[wave * MXE_PARTS + part] = vu;
    lds_barrier();
    if (tid < 32) gates[tid] = silu_as_host(gates[tid], table) * ups[tid];
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the wavefront's own LDS)
    if (tid < 8) {
        uint32_t q;
        const float d = quantize(reinterpret_cast<const float4 *>(gates)[tid], q);
        reinterpret_cast<uint32_t *>(g.q + (size_t)pair * g.ffn + (size_t)blockIdx.x * 32)[tid] = q;
        if (tid == 0) g.d[(size_t)pair * (g.ffn / 32) + blockIdx.x] = d;
    }
#endif
}

struct MxeDownArgs {
    const uint8_t *W;
    size_t row_stride;
    int rows, units, n_experts, k, rows_wg;
    const int32_t *ids;
    const float *weights;
    const int8_t *q;
    const float *d;
    float *out;  // [token][rows]
};
template <int S>
__global__ __launch_bounds__(64 * MXE_WAVES, 3) void mx_experts_down_kernel(MxeDownArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
    __shared__ float sums[MXE_MAX_SLOTS * MXE_MAX_ROWS], slot_weight[MXE_MAX_SLOTS];
    __shared__ int slot_id[MXE_MAX_SLOTS];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), waves = (int)blockDim.x >> 6;
    const int l = lane % MXE_LANES, part = lane / MXE_LANES, units = g.units;
    const size_t first = (size_t)blockIdx.y * g.k;
    const int row_begin = (int)blockIdx.x * g.rows_wg, row_end = min(g.rows, row_begin + g.rows_wg);
    const bool lists = tid < g.k;
    const int list_id = lists ? g.ids[first + tid] : 0;
    const float list_weight = lists ? g.weights[first + tid] : 0.0f;
    for (int slot = wave; slot < g.k; slot += waves) {
        const int id = __builtin_amdgcn_readfirstlane(g.ids[first + slot]);
        if (id < 0 || id >= g.n_experts) continue;  // (left out of the sum)
        const uint8_t *We = g.W + (size_t)id * g.rows * g.row_stride;
        MxeRow<S> w;
        auto request = [&](int r0) { w.load(We + (size_t)min(r0 + part, g.rows - 1) * g.row_stride, l, units); };
        request(row_begin);
        const uint4 *const qs = reinterpret_cast<const uint4 *>(g.q + (first + slot) * (size_t)units * 32);
        const float *const ds = g.d + (first + slot) * (size_t)units;
        uint4 a[S], b[S];
        float d[S];
#pragma unroll
        for (int s = 0; s < S; s++) {
            const int at = min(l + s * MXE_LANES, units - 1);
            a[s] = qs[2 * at], b[s] = qs[2 * at + 1], d[s] = ds[at];
        }
        for (int r0 = row_begin; r0 < row_end; r0 += MXE_PARTS) {
            const MxeRow<S> now = w;
            if (r0 + MXE_PARTS < row_end) request(r0 + MXE_PARTS);
            float t[S];
#pragma unroll
            for (int s = 0; s < S; s++) t[s] = l + s * MXE_LANES < units ? now.term(s, a[s], b[s], d[s]) : 0.0f;
            const float v = mxe_sum(t);
            if (l == 0 && r0 + part < row_end) sums[slot * g.rows_wg + r0 + part - row_begin] = v;
        }
    }
    if (lists) slot_id[tid] = list_id, slot_weight[tid] = list_weight;
    __syncthreads();
    const int r = row_begin + tid;
    if (tid < g.rows_wg && r < row_end) {
        float acc = 0.0f;
        for (int s = 0; s < g.k; s++) {  // in routing order (combine_expert_outputs), a multiply and an add each
            const int id = slot_id[s];
            if (id >= 0 && id < g.n_experts) acc += slot_weight[s] * sums[s * g.rows_wg + tid];
        }
        g.out[(size_t)blockIdx.y * g.rows + r] = acc;
    }
#endif
}

// Rows of a down workgroup: four a wavefront's turn, as many turns as leave 16 wavefronts a CU
static int mxe_rows_wg(size_t rows, size_t batch, int waves) {
    const size_t turns = rows * batch * (size_t)waves / (MXE_PARTS * 16 * 256);
    return MXE_PARTS * (int)std::min<size_t>(std::max<size_t>(turns, 1), MXE_MAX_ROWS / MXE_PARTS);
}

bool mx_experts_take(const frk_weights *gate, const frk_weights *up, const frk_weights *down, size_t batch, size_t k) {
    return gate->kind == FRK_KIND_MXFP4 && up->kind == FRK_KIND_MXFP4 && down->kind == FRK_KIND_MXFP4 && gate->cols <= 32 * MXE_MAX_UNITS &&
           down->cols <= 32 * MXE_MAX_UNITS && gate->layout.row_stride == up->layout.row_stride && k <= MXE_MAX_SLOTS && batch * k <= 65535;
}

// q, d: room for the pairs' quantized intermediate
int launch_mx_experts(const frk_weights *gate, const frk_weights *up, const frk_weights *down, int n_experts, const float *x, size_t batch,
                      const int32_t *ids, const float *weights, int k, int8_t *q, float *d, float *out, hipStream_t s) {
    const int hidden = (int)gate->cols, ffn = (int)down->cols;
    const MxeGateUpArgs ga{gate->dev, up->dev, gate->layout.row_stride, ffn, hidden / 32, n_experts, k, ids, x, q, d};
    const dim3 grid_a((unsigned)(ffn / 32), (unsigned)(batch * (size_t)k));
#define FRK_GO(KERNEL, UNITS, GRID, THREADS, ARGS)                                                          \
    switch (((UNITS) + MXE_LANES - 1) / MXE_LANES) {                                                        \
    case 1:                                                                                                 \
    case 2: hipLaunchKernelGGL(KERNEL<2>, GRID, dim3(THREADS), 0, s, ARGS); break;                          \
    case 3: hipLaunchKernelGGL(KERNEL<3>, GRID, dim3(THREADS), 0, s, ARGS); break;                          \
    case 4: hipLaunchKernelGGL(KERNEL<4>, GRID, dim3(THREADS), 0, s, ARGS); break;                          \
    case 5: hipLaunchKernelGGL(KERNEL<5>, GRID, dim3(THREADS), 0, s, ARGS); break;                          \
    default: hipLaunchKernelGGL(KERNEL<6>, GRID, dim3(THREADS), 0, s, ARGS);                                \
    }                                                                                                       \
    {                                                                                                       \
        const hipError_t e = hipGetLastError();                                                             \
        if (e != hipSuccess) return set_error(FRK_ERR_HIP, #KERNEL " launch: %s", hipGetErrorString(e));    \
    }
    FRK_GO(mx_experts_gate_up_kernel, hidden / 32, grid_a, 512, ga)
    const int waves = std::min(k, MXE_WAVES), rows_wg = mxe_rows_wg((size_t)hidden, batch, waves);
    const MxeDownArgs da{down->dev, down->layout.row_stride, hidden, ffn / 32, n_experts, k, rows_wg, ids, weights, q, d, out};
    const dim3 grid_d((unsigned)((hidden + rows_wg - 1) / rows_wg), (unsigned)batch);
    FRK_GO(mx_experts_down_kernel, ffn / 32, grid_d, 64 * waves, da)
#undef FRK_GO
    return FRK_OK;
}

}  // namespace frk
