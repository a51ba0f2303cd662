// Activations for the MXFP4 experts on the block-scaled matrix cores (frk_gemm_mx.hip): Q8_0 blocks as planes of digits.
#pragma once

#include "frk_device.hpp"

namespace frk {

// ---- activations: rows of blocks, a row padded with zero blocks to a multiple of eight.  A block: six 16-byte pieces --
// dwords 0..3 of the planes 0..3, dwords 4 and 5 of planes 0 and 1, of planes 2 and 3 -- and one dword of the four planes'
// E8M0 scales.  Four blocks' pieces lie together: the four first ones, the four second ones, ... ----
constexpr int MX_BLOCK_BYTES = 96;
static __host__ __device__ inline size_t mx_padded_blocks(size_t cols) { return (cols / 32 + 7) / 8 * 8; }

// |v| <= 127 * 2047 as four signed base-32 digits, digit p's E2M3 code in byte p.  With 16 added at every place the digits
// are the number's own bits; x = digit + 16 (0 .. 31) a byte each, then four codes at a time: the magnitude a = |x - 16| in
// units of a quarter is 2a up to 7 and a + 8 from 8 on, under the sign.
__device__ __forceinline__ uint32_t mx_digit_codes(int v) {
    const uint32_t u = (uint32_t)(v + 16 * (1 + 32 + 32 * 32 + 32 * 32 * 32));
    const uint32_t t = (u & 0x3ffu) | ((u << 6) & 0x03ff0000u);
    const uint32_t x = (t & 0x001f001fu) | ((t << 3) & 0x1f001f00u);
    const uint32_t n = (~x >> 4) & 0x01010101u;                                    // negative
    const uint32_t a = ((x & 0x0f0f0f0fu) ^ ((n << 5) - n)) - ((n << 4) - n);      // n: (31 - low) - 15
    const uint32_t g = ((a >> 3) | (a >> 4)) & 0x01010101u;                        // 8 or more
    return (a + ((a & (0x07070707u ^ ((g << 3) - g))) | (g << 3))) | (n << 5);
}

// quantize_activations_q8, Avx form (crates/frink-quant/src/act_quant.rs:157-189), and the digits of quant * scale.
// `threads` threads (tid; whole wavefronts) of a workgroup per row, four lanes per block, a lane elements 4i .. 4i+3 and 16+4i .. 16+4i+3: eight
// neighbours in the digits' order, 48 bits of a plane.  `flag`: a word of LDS per row, zero before; a workgroup's rows meet
// at one barrier.
// A block whose scale overflows f16 (a largest value above 8.3e6; its E8M0 bytes start at MX_INFINITE) makes an infinity of
// its integer sum, NaN where that is zero.  A row with such blocks is marked in `infinite`, and they keep their 32 quants as
// bytes where the digits of a block would start: the GEMM ends with such rows on their own.
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
    auto quant = [&](int i) {
        const float r = rintf(e[i] * inv);
        return (r != r) ? 0 : (int)fminf(fmaxf(r, -127.0f), 127.0f);
    };
    int infinite = 0;
    for (int b = tid >> 2; b < nbp; b += threads >> 2) {
        const uint32_t d = load(b);
        const int ex = (int)(d >> 10), mant = (int)(d & 1023u) | (ex ? 1024 : 0);
        infinite |= ex == 31;
        uint32_t codes[8];  // an element's four digits' codes, plane p in byte p
#pragma unroll
        for (int i = 0; i < 8; i++) codes[i] = mx_digit_codes(quant(i) * mant);
        uint32_t low[4], high[4];  // a plane's 48 bits
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t *c = codes + 4 * h;
            const uint32_t a01 = __builtin_amdgcn_perm(c[1], c[0], 0x05010400u), b01 = __builtin_amdgcn_perm(c[1], c[0], 0x07030602u);
            const uint32_t a23 = __builtin_amdgcn_perm(c[3], c[2], 0x05010400u), b23 = __builtin_amdgcn_perm(c[3], c[2], 0x07030602u);
            const uint32_t by_plane[4] = {__builtin_amdgcn_perm(a23, a01, 0x05040100u), __builtin_amdgcn_perm(a23, a01, 0x07060302u),
                                          __builtin_amdgcn_perm(b23, b01, 0x05040100u), __builtin_amdgcn_perm(b23, b01, 0x07060302u)};
#pragma unroll
            for (int p = 0; p < 4; p++) {
                const uint32_t w = by_plane[p];
                const uint32_t bits24 = (w & 0x3fu) | ((w >> 2) & 0xfc0u) | ((w >> 4) & 0x3f000u) | ((w >> 6) & 0xfc0000u);
                if (h == 0) low[p] = bits24;
                else low[p] |= bits24 << 24, high[p] = bits24 >> 8;
            }
        }
        // lanes in pairs: the even one writes planes 0 and 1 of the pair's 96 bits, the odd one planes 2 and 3
        const bool odd = part & 1;
        const size_t at = (size_t)row * nbp + b;
        uint32_t *dst = reinterpret_cast<uint32_t *>(out.digits + (at & ~(size_t)3) * MX_BLOCK_BYTES) + (b & 3) * 4;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const uint32_t own_low = odd ? low[2 + h] : low[h], own_high = odd ? high[2 + h] : high[h];
            const uint32_t other_low = (uint32_t)dpp_i<DPP_QUAD_XOR1>((int)(odd ? low[h] : low[2 + h]));
            const uint32_t other_high = (uint32_t)dpp_i<DPP_QUAD_XOR1>((int)(odd ? high[h] : high[2 + h]));
            const uint32_t first_low = odd ? other_low : own_low, first_high = odd ? other_high : own_high;
            const uint32_t second_low = odd ? own_low : other_low, second_high = odd ? own_high : other_high;
            const uint32_t w[3] = {first_low, first_high | (second_low << 16), (second_low >> 16) | (second_high << 16)};
            const int p = (odd ? 2 : 0) + h;
#pragma unroll
            for (int k = 0; k < 3; k++) {
                const int j = 3 * (part >> 1) + k;
                dst[j < 4 ? 16 * p + j : 64 + 16 * (p >> 1) + 2 * (p & 1) + j - 4] = w[k];
            }
        }
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
                return (uint32_t)(quant(i) & 0xff) | (uint32_t)(quant(i + 2) & 0xff) << 8 | (uint32_t)(quant(i + 4) & 0xff) << 16 | (uint32_t)(quant(i + 6) & 0xff) << 24;
            };
            uint32_t *dst = reinterpret_cast<uint32_t *>(out.digits + ((size_t)row * nbp + b) * MX_BLOCK_BYTES);
            dst[part] = bytes(0), dst[4 + part] = bytes(1);
        }
    if (tid == 0) out.infinite[row] = row_infinite;
}

}  // namespace frk
