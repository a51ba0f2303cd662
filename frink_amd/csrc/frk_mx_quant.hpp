// Activations for the MXFP4 experts on the block-scaled matrix cores (frk_gemm_mx.hip): Q8_0 blocks as planes of digits.
#pragma once

#include "frk_device.hpp"

namespace frk {

// ---- activations: rows of blocks, a row padded with zero blocks to a multiple of eight.  A block: six 16-byte pieces --
// dwords 0..3 of the planes 0..3, dwords 4 and 5 of planes 0 and 1, of planes 2 and 3 -- and one dword of the four planes'
// E8M0 scales.  Four blocks' pieces lie together: the four first ones, the four second ones, ... ----
constexpr int MX_BLOCK_BYTES = 96;
static __host__ __device__ inline size_t mx_padded_blocks(size_t cols) { return (cols / 32 + 7) / 8 * 8; }

typedef _Float16 mx_v32h __attribute__((ext_vector_type(32)));
typedef uint32_t mx_v6u __attribute__((ext_vector_type(6)));

// Eight numbers, |v| <= 127 * 2047, as four signed base-32 digits each: 48 bits of E2M3 codes a plane, in units of a quarter.
// (In units of an eighth the codes would be the digits' magnitudes, but the matrix core drops low places of such products
// sooner: up to 1.12 times the error against 64 bits.)  With 16 added at every place the digits are the number's own bits, 0 ..
// 31 each; as the bits of an f16 those are multiples of 2^-24, from which 16 are taken away again and 32 digits go through one
// conversion, all exact.
__device__ __forceinline__ mx_v6u mx_digit_codes(const int v[8]) {
    uint32_t digits[4][4];  // [plane][two numbers]
#pragma unroll
    for (int j = 0; j < 4; j++) {
        constexpr int EACH = 16 * (1 + 32 + 32 * 32 + 32 * 32 * 32);
        const uint32_t u0 = (uint32_t)(v[2 * j] + EACH), u1 = (uint32_t)(v[2 * j + 1] + EACH);
        const uint32_t low = __builtin_amdgcn_perm(u1, u0, 0x05040100u), high = __builtin_amdgcn_perm(u1, u0, 0x06050201u);  // bits 0 .. 15, 8 .. 23
        digits[0][j] = low & 0x001f001fu, digits[1][j] = (low >> 5) & 0x001f001fu;
        digits[2][j] = (high >> 2) & 0x001f001fu, digits[3][j] = (high >> 7) & 0x001f001fu;
    }
    mx_v32h all;
    __builtin_memcpy(&all, digits, sizeof all);
    const _Float16 sixteen = (_Float16)(16.0f / 16777216.0f);
    all -= sixteen;
    return __builtin_amdgcn_cvt_scalef32_pk32_fp6_f16(all, 4.0f / 16777216.0f);
}

// quantize_activations_q8, Avx form (crates/frink-quant/src/act_quant.rs:157-189), and the digits of quant * scale.
// `threads` threads (tid; whole wavefronts) of a workgroup per row, four lanes per block, a lane elements 4i .. 4i+3 and 16+4i .. 16+4i+3: eight
// neighbours in the digits' order, 48 bits of a plane.  `flag`: a word of LDS per row, zero before; a workgroup's rows meet
// at one barrier.
// A block whose scale overflows f16 (a largest value above 8.3e6; its E8M0 bytes start at MX_INFINITE) makes an infinity of
// its integer sum, NaN where that is zero.  A row with such blocks is marked in `infinite`, and they keep their 32 quants as
// bytes where the digits of a block would start: the GEMM ends with such rows on their own.
// The vector ALU bounds it (41 MB for 2048 rows of 2880 columns, 8.7 us at a copy's rate): 18.9 us under the profiler with every
// code made and packed by integer instructions, a float clamp and stores of single dwords, 11.6 so; 32 experts top-4 of 2880 / 2880 at
// 512 tokens, the layer, 240 -> 230.  The same codes.
constexpr uint32_t MX_INFINITE = 31 + 104;
__device__ __forceinline__ void quantize_mx_row(const float *__restrict__ x, int row, int nb, int tid, int threads, int *flag, const MxActs &out) {
    const int nbp = (nb + 7) & ~7, part = tid & 3;
    const float *xr = x + (size_t)row * nb * 32;
    float e[8];  // this lane's elements of a block
    float inv;   // 1 / scale
    auto load = [&](int b) {  // the block's f16 scale
        float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
        if (b < nb) {
            lo = reinterpret_cast<const float4 *>(xr + b * 32)[part];
            hi = reinterpret_cast<const float4 *>(xr + b * 32)[4 + part];
        }
        e[0] = lo.x, e[1] = hi.x, e[2] = lo.y, e[3] = hi.y, e[4] = lo.z, e[5] = hi.z, e[6] = lo.w, e[7] = hi.w;
        float amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(e[i]));
        amax = fmaxf(amax, dpp_f<DPP_QUAD_XOR1>(amax));
        amax = fmaxf(amax, dpp_f<DPP_QUAD_XOR2>(amax));
        inv = amax != 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
        return f2h_bits(__fdiv_rn(amax, 127.0f));
    };
    auto quant = [&](int i) { return quant_of(e[i] * inv); };
    int infinite = 0;
    for (int b = tid >> 2; b < nbp; b += threads >> 2) {
        const uint32_t d = load(b);
        const int ex = (int)(d >> 10), mant = (int)(d & 1023u) | (ex ? 1024 : 0);
        infinite |= ex == 31;
        int v[8];
#pragma unroll
        for (int i = 0; i < 8; i++) v[i] = quant(i) * mant;
        const mx_v6u own = mx_digit_codes(v);  // a plane's 48 bits after the other's
        // lanes in pairs: the even one has planes 0 and 1 of the pair's 96 bits, the odd one planes 2 and 3
        const bool odd = part & 1;
        const size_t at = (size_t)row * nbp + b;
        uint32_t first[3], second[3];  // the even lane's share of the two planes, the odd lane's
#pragma unroll
        for (int k = 0; k < 3; k++) {
            uint32_t low = own[k], high = own[3 + k];
            asm("" : "+v"(low), "+v"(high));  // (else a choice of index, and a chain of compares)
            const uint32_t from_even = (uint32_t)dpp_i<DPP_QUAD_XOR1>((int)high), from_odd = (uint32_t)dpp_i<DPP_QUAD_XOR1>((int)low);
            first[k] = odd ? from_even : low, second[k] = odd ? high : from_odd;
        }
        const uint32_t w[2][3] = {{first[0], (first[1] & 0xffffu) | (second[0] << 16), (second[0] >> 16) | (second[1] << 16)},
                                  {(first[1] >> 16) | (first[2] << 16), (first[2] >> 16) | (second[1] & 0xffff0000u), second[2]}};
        // (lanes 0 and 1 have dwords 0..2, 2 and 3 dwords 3..5: whole pieces from each)
        const uint32_t third0 = (uint32_t)dpp_i<DPP_QUAD_XOR2>((int)w[0][0]), third1 = (uint32_t)dpp_i<DPP_QUAD_XOR2>((int)w[1][0]);
        uint4 *dst = reinterpret_cast<uint4 *>(out.digits + (at & ~(size_t)3) * MX_BLOCK_BYTES) + (b & 3);
        const bool tail = part & 2;
        dst[4 * (tail ? 4 + (part & 1) : 2 * part)] =
            tail ? make_uint4(w[0][1], w[0][2], w[1][1], w[1][2]) : make_uint4(w[0][0], w[0][1], w[0][2], third0);
        if (!tail) dst[4 * (2 * part + 1)] = make_uint4(w[1][0], w[1][1], w[1][2], third1);
        // 2^(ex - 25) a unit, a digit's code is a quarter of its value, plane p times 32^p
        if (part == 0) out.scales[at] = 0x0f0a0500u + 0x01010101u * (uint32_t)(max(ex, 1) + 104);
    }
    if (infinite) *flag = 1;
    __syncthreads();
    const bool row_infinite = *flag != 0;
    if (row_infinite)  // (over digits of the row that nobody will look at)
        for (int b = tid >> 2; b < nb; b += threads >> 2) {
            if (load(b) >> 10 != 31) continue;
            auto bytes = [&](int i) {
                return quants_of(quant(i), quant(i + 2), quant(i + 4), quant(i + 6));
            };
            uint32_t *dst = reinterpret_cast<uint32_t *>(out.digits + ((size_t)row * nbp + b) * MX_BLOCK_BYTES);
            dst[part] = bytes(0), dst[4 + part] = bytes(1);
        }
    if (tid == 0) out.infinite[row] = row_infinite;
}

}  // namespace frk
