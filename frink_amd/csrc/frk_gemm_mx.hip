// Grouped GEMM over MXFP4 experts on the block-scaled matrix cores (v_mfma_scale_f32_32x32x64_f8f6f4):
//   y[token][row] = sum over the 32-wide blocks of  (dw * da) * sum_i qw_i * qa_i
// with the activations quantized to Q8_0 blocks as on every integer path of this kind (dot_mxfp4_q8,
// crates/frink-quant/src/legacy_q8.rs:169-213; the MoE bucket path, crates/frink-models/src/decoder/ffn_batch.rs:343-434).
//
// The matrix core takes an MXFP4 block as it is stored: sixteen bytes of E2M1 codes are a lane's operand, the block's
// E8M0 byte its scale.  The activation block's  da * qa  is a 19-bit number (f16 scale: 11 bits of mantissa, 8-bit quant)
// times a power of two, and goes through as four planes of signed base-32 digits, -16 .. 16: exact in E2M3 (six bits),
// the power of two and the plane's 32^p in its E8M0 scale.  So every product is exact, sums are f32 inside the matrix
// core, and the vector ALU has no float step at all -- it adds the sums of 128 columns onto the running ones, which keeps
// the error against 64 bits below that of one addition a block (2-norm over 2-norm at 1024 / 1184 / 2048 columns: 5.8e-8,
// 6.2e-8 and 7.9e-8, with an addition a block 7.6e-8, 8.2e-8 and 1.1e-7).
// (Byte i of a GGUF block holds elements i and i + 16; a lane's operand takes byte i as k = 2i and 2i + 1.  The order of
// k within a block is free as long as both operands have it: the digits are stored in the weights' order.)
//
// Before, the experts were decoded to signed bytes with f16 scales on every call (83 us a projection of 32 x 2880 x
// 2880) and multiplied by the Q8_0 kernel, whose float step is 32 vector instructions per MFMA (156 us).
#include "frk_device.hpp"

#include <type_traits>

namespace frk {

typedef int mx_v4i __attribute__((ext_vector_type(4)));
typedef int mx_v8i __attribute__((ext_vector_type(8)));
typedef float mx_v16f __attribute__((ext_vector_type(16)));

#define FRK_LAUNCH_CHECK(what)                                                                          \
    do {                                                                                                \
        hipError_t e_ = hipGetLastError();                                                              \
        if (e_ != hipSuccess) return set_error(FRK_ERR_HIP, what " launch: %s", hipGetErrorString(e_)); \
    } while (0)

// ---- activations: rows of blocks, a row padded with zero blocks to a multiple of eight.  A block: six 16-byte pieces --
// dwords 0..3 of the planes 0..3, dwords 4 and 5 of planes 0 and 1, of planes 2 and 3 -- and one dword of the four planes'
// E8M0 scales.  Four blocks' pieces lie together: the four first ones, the four second ones, ... ----
constexpr int MX_BLOCK_BYTES = 96;
static __host__ __device__ inline size_t mx_padded_blocks(size_t cols) { return (cols / 32 + 7) / 8 * 8; }

MxActs mx_acts_carve(void *base, size_t rows, size_t cols) {
    const size_t blocks = rows * mx_padded_blocks(cols);
    MxActs a;
    a.digits = (uint8_t *)base;
    a.scales = (uint32_t *)((char *)base + round_up(blocks * MX_BLOCK_BYTES, 256));
    a.factor = (float *)((char *)a.scales + round_up(blocks * 4, 256));
    return a;
}
size_t mx_acts_bytes(size_t rows, size_t cols) {
    const size_t blocks = rows * mx_padded_blocks(cols);
    return round_up(blocks * MX_BLOCK_BYTES, 256) + round_up(blocks * 4, 256) + round_up(rows * 4, 256);
}

// quantize_activations_q8, Avx form (crates/frink-quant/src/act_quant.rs:157-189), and the digits of quant * scale.
// A workgroup per row, four lanes per block, a lane elements 4i .. 4i+3 and 16+4i .. 16+4i+3: eight neighbours in the
// digits' order, 48 bits of a plane.  `used`: a row whose entry is negative is left as it is.
// A block whose scale overflows f16 (a largest value above 8.3e6) makes the row's results infinite (NaN where its sum
// is zero): its digits are kept with a scale of 65536, the row's other blocks are zeroed, and `factor` carries the
// infinity to the end.
__global__ __launch_bounds__(128) void quantize_mx_kernel(const float *__restrict__ x, int nb, const int *__restrict__ used, MxActs out) {
    const int row = blockIdx.x;
    if (used && used[row] < 0) return;
    const int nbp = (nb + 7) & ~7, part = threadIdx.x & 3;
    const float *xr = x + (size_t)row * nb * 32;
    bool row_infinite = false;
    for (int pass = 0; pass < 2; pass++) {
        int infinite = 0;
        for (int b = threadIdx.x >> 2; b < nbp; b += 32) {
            float4 lo = make_float4(0.f, 0.f, 0.f, 0.f), hi = lo;
            if (b < nb) {
                lo = reinterpret_cast<const float4 *>(xr + b * 32)[part];
                hi = reinterpret_cast<const float4 *>(xr + b * 32)[4 + part];
            }
            const float e[8] = {lo.x, hi.x, lo.y, hi.y, lo.z, hi.z, lo.w, hi.w};
            float amax = 0.0f;
#pragma unroll
            for (int i = 0; i < 8; i++) amax = fmaxf(amax, fabsf(e[i]));
            amax = fmaxf(amax, __shfl_xor(amax, 1));
            amax = fmaxf(amax, __shfl_xor(amax, 2));
            const float inv = amax != 0.0f ? __fdiv_rn(127.0f, amax) : 0.0f;
            const uint32_t d = f2h_bits(__fdiv_rn(amax, 127.0f));
            const int ex = (int)(d >> 10);
            int mant = (int)(d & 1023u) | (ex ? 1024 : 0);
            infinite |= ex == 31;
            if (pass && ex != 31) mant = 0;
            uint64_t planes[4] = {0, 0, 0, 0};
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float r = rintf(e[i] * inv);
                int v = ((r != r) ? 0 : (int)fminf(fmaxf(r, -127.0f), 127.0f)) * mant;
#pragma unroll
                for (int p = 0; p < 4; p++) {
                    const int digit = ((v + 16) & 31) - 16;
                    v = (v - digit) >> 5;
                    const int a = abs(digit);
                    // E2M3 in units of a quarter: 0 .. 7 are 2a, 8 .. 16 are a + 8
                    const uint32_t code = (uint32_t)(a < 8 ? 2 * a : a + 8) | (digit < 0 ? 32u : 0u);
                    planes[p] |= (uint64_t)code << (6 * i);
                }
            }
            // lanes in pairs: the even one writes planes 0 and 1 of the pair's 96 bits, the odd one planes 2 and 3
            const bool odd = part & 1;
            const size_t at = (size_t)row * nbp + b;
            uint32_t *dst = reinterpret_cast<uint32_t *>(out.digits + (at & ~(size_t)3) * MX_BLOCK_BYTES) + (b & 3) * 4;
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint64_t own = odd ? planes[2 + h] : planes[h];
                const uint64_t other = __shfl_xor((unsigned long long)(odd ? planes[h] : planes[2 + h]), 1);
                const uint64_t first = odd ? other : own, second = odd ? own : other;
                const uint32_t w[3] = {(uint32_t)first, (uint32_t)(first >> 32) | (uint32_t)(second << 16), (uint32_t)(second >> 16)};
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
        if (pass) break;
        row_infinite = __syncthreads_or(infinite) != 0;
        if (!row_infinite) break;
    }
    if (threadIdx.x == 0) out.factor[row] = row_infinite ? __builtin_inff() : 1.0f;
}
int launch_quantize_mx(const float *x, size_t rows, size_t cols, const int *used, const MxActs &out, hipStream_t s) {
    if (rows == 0) return FRK_OK;
    hipLaunchKernelGGL(quantize_mx_kernel, dim3((unsigned)rows), dim3(128), 0, s, x, (int)(cols / 32), used, out);
    FRK_LAUNCH_CHECK("quantize_mx");
    return FRK_OK;
}

// ---- the GEMM.  A workgroup of NW wavefronts multiplies one tile (at most 64 activation rows of one group, two halves
// of 32) with 64 weight rows a wavefront, as two groups of 32: of one matrix, or (GLU) the same rows of gate and up,
// whose results meet in the epilogue as silu(gate) * up.
//
// The columns go by four blocks at a time: step s (0, 1) multiplies blocks s and 2 + s, a lane block s or 2 + s of its
// row by its half (k = 64).  Everything comes straight into LDS: the activations' digits (25 KB) two quads of blocks ahead
// in a ring of three stages that the workgroup shares, with one barrier a quad; the weights one quad ahead into a
// wavefront's own two slots, their scale bytes four quads at a time.
// What bounds the kernel is the way of those bytes into LDS (60 KB a quad of 2048 clocks of matrix core): neighbouring
// lanes of a request fetch neighbouring pieces of memory (384 bytes of digits, 64 of codes a row), the LDS images are
// swizzled so that a fragment's reads -- one piece of sixteen rows each -- fall in different banks, and the requests are
// spread over the quad's arithmetic.  Gate and up of 32 experts of 2880 x 2880 over 2048 pairs: weights loaded into
// registers, a row a lane, 227 us; weights in LDS but a lane per activation row 208 us; as it is now 171 us (the bytes
// from memory take 50, the matrix core 40).  Eight wavefronts a workgroup where that still fills the chip: a stage of
// digits then serves twice the rows (the down projection 137 -> 96 us). ----
struct MxGemmArgs {
    const uint8_t *W, *W2;  // GLU: gate and up
    size_t row_stride, group_stride;
    int rows, nb;  // of one group
    MxActs acts;
    const int *src_rows;  // the activation row of a row of the grouped order (negative: none); null: the row itself
    const int4 *tiles;    // {group, first row of the grouped order, rows in use, first row of y}
    const int *n_tiles;
    int row_groups;  // workgroups a tile
    float *y;
};
constexpr int MX_ROW = 4 * MX_BLOCK_BYTES;             // an activation row's digits of one quad, 24 pieces
constexpr int MX_STAGE_SCALES = 64 * MX_ROW;           // [64 rows][4 blocks] dwords
constexpr int MX_STAGE = MX_STAGE_SCALES + 64 * 16;
constexpr int MX_STAGES = 3;
constexpr int MX_W_SCALES = 2 * 4096;                  // two slots of codes [64 rows][4 blocks], two of scales [64 rows][16]
constexpr int MX_W_WAVE = MX_W_SCALES + 2 * 1024;
template <int NW>
constexpr size_t mx_lds_bytes() { return (size_t)MX_STAGES * MX_STAGE + (size_t)NW * MX_W_WAVE; }
static_assert(mx_lds_bytes<8>() <= 160 * 1024, "LDS of a CU");

template <int NW, bool GLU>
__global__ __launch_bounds__(64 * NW, 2) void gemm_mx_grouped_kernel(MxGemmArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
    extern __shared__ __align__(16) uint8_t mx_lds[];
    uint8_t *const lds = mx_lds;
    // the workgroups of a tile sit on one XCD (block id mod 8), whose L2 then serves the tile's digits
    const int j = (int)blockIdx.x >> 3, t = ((int)blockIdx.x & 7) + 8 * (j / g.row_groups);
    if (t >= *g.n_tiles) return;
    const int4 tile = g.tiles[t];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int li = lane & 31, lg = lane >> 5;
    const int nb = g.nb, nbp = (nb + 7) & ~7;
    const int quads = (nb + 3) >> 2;
    const bool two = tile.z > 32;

    const uint32_t lds0 = lds_address(lds);
    // ---- weights: rows row0 + lane % 32 of the two groups.  Request c of a quad brings rows 16c .. 16c + 15 of the 64:
    // slot p of row r holds block p ^ (r / 4) % 4, so that the reads of one block of 32 rows fall in different banks.
    const int row_wave = ((j % g.row_groups) * NW + wave) * (GLU ? 32 : 64), row0 = row_wave + li;
    const uint8_t *const w_base[2] = {g.W + (size_t)tile.x * g.group_stride, (GLU ? g.W2 : g.W) + (size_t)tile.x * g.group_stride};
    auto weight_row = [&](int r) {  // row r of the wavefront's 64 as a row of its matrix
        return (uint32_t)min(GLU ? row_wave + (r & 31) : row_wave + r, g.rows - 1) * (uint32_t)g.row_stride;
    };
    uint32_t codes_off[4];
#pragma unroll
    for (int c = 0; c < 4; c++)
        codes_off[c] = weight_row(16 * c + (lane >> 2)) + (uint32_t)((lane & 3) ^ ((lane >> 4) & 3)) * 16;
    const uint32_t w_scales_off = weight_row(lane);
    const uint32_t w_lds = lds0 + MX_STAGES * MX_STAGE + (uint32_t)wave * MX_W_WAVE;
    // (a row's last quad may reach past the row, by less than 64 bytes: the resident copy ends in 256 bytes of slack.
    // What those bytes hold meets zero digits, its scale byte is not used.)
    auto fetch_codes = [&](int i, int c) {  // request c of quad i
        dma16(w_lds + (uint32_t)(i & 1) * 4096 + c * 1024, w_base[c >> 1] + (size_t)i * 64, codes_off[c]);
    };
    auto fetch_weight_scales = [&](int i) {  // of quads i .. i + 3
        const uint32_t to = w_lds + MX_W_SCALES + (uint32_t)((i >> 2) & 1) * 1024;
        const size_t at = (size_t)nb * 16 + (size_t)i * 4;
        if (!GLU || lane < 32) dma16(to, w_base[0] + at, w_scales_off);
        else dma16(to, w_base[1] + at, w_scales_off);
    };

    // ---- activations: a stage's digits are 64 rows of 24 pieces, piece s of row r in place s ^ (r / 2) % 8 (sixteen rows reading one
    // piece each then touch sixteen different pieces of the 64 banks); each wavefront
    // fetches its share of the 24 requests, the first one the scales too
    constexpr int REQUESTS = 24 / NW;
    static_assert(24 % NW == 0, "whole requests");
    auto act_row = [&](int r) { return (uint32_t)(g.src_rows ? max(g.src_rows[tile.y + r], 0) : tile.y + r); };
    uint32_t digits_off[REQUESTS];
#pragma unroll
    for (int c = 0; c < REQUESTS; c++) {
        const int at = (wave * REQUESTS + c) * 64 + lane, r = at / 24;
        digits_off[c] = act_row(r) * (uint32_t)nbp * MX_BLOCK_BYTES + (uint32_t)((at % 24) ^ ((r >> 1) & 7)) * 16;
    }
    const uint32_t scales_off = act_row(lane) * (uint32_t)nbp * 4;
    auto fetch_digits = [&](int i, int c) {
        dma16(lds0 + (uint32_t)(i % MX_STAGES) * MX_STAGE + (uint32_t)(wave * REQUESTS + c) * 1024, g.acts.digits + (size_t)i * MX_ROW,
              digits_off[c]);
    };
    auto fetch_act_scales = [&](int i) {
        if (wave == 0) dma16(lds0 + (uint32_t)(i % MX_STAGES) * MX_STAGE + MX_STAGE_SCALES, g.acts.scales + (size_t)i * 4, scales_off);
    };
    // What a wavefront requests during quad i, in four portions (the address unit takes a clock per lane of a request:
    // all at once, the requests of eight wavefronts hold each other up for longer than the quad's arithmetic takes):
    // the weights of quad i + 1, then the digits of quad i + 2.
    auto request = [&](auto portion_c, int i) {
        constexpr int P = decltype(portion_c)::value;
        if (P < 2 && i + 1 < quads) {
            fetch_codes(i + 1, 2 * P);
            fetch_codes(i + 1, 2 * P + 1);
            if (P == 1 && ((i + 1) & 3) == 0) fetch_weight_scales(i + 1);
        }
        if (P >= 2 && i + 2 < quads) {
#pragma unroll
            for (int c = (P - 2) * ((REQUESTS + 1) / 2); c < (P == 2 ? (REQUESTS + 1) / 2 : REQUESTS); c++) fetch_digits(i + 2, c);
            if (P == 3) fetch_act_scales(i + 2);
        }
    };
    // where this lane's pieces of step k sit in a half's 32 rows: piece 4n + block in place (4n + block) ^ x, so the even n
    // 128 bytes apart from here, the odd ones from there
    uint32_t piece_at[2][2];
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int n = 0; n < 2; n++) piece_at[k][n] = (uint32_t)(li * MX_ROW + ((4 * n + 2 * lg + k) ^ ((li >> 1) & 7)) * 16);

    mx_v16f acc[2][2];  // [half][row group]
#pragma unroll
    for (int h = 0; h < 2; h++)
#pragma unroll
        for (int r = 0; r < 2; r++) acc[h][r] = mx_v16f{0.0f};

    // one quad: per half two steps of four planes of digits, smallest first, their sum added onto the running one; a
    // step's operands are read while the one before is multiplied
    auto multiply = [&](int i) {
        constexpr int E2M3 = 2, E2M1 = 4;
        const uint8_t *st = lds + (size_t)(i % MX_STAGES) * MX_STAGE;
        const uint8_t *w_wave = lds + MX_STAGES * MX_STAGE + (size_t)wave * MX_W_WAVE, *ws = w_wave + (i & 1) * 4096;
        const uint8_t *w_scales = w_wave + MX_W_SCALES + ((i >> 2) & 1) * 1024 + (i & 3) * 4;
        // the codes of step k and row group r, and the scale bytes of the lane's two blocks (a block past the row's end: 2^-127)
        auto codes = [&](int k, int r) {
            const mx_v4i v = *reinterpret_cast<const mx_v4i *>(ws + (32 * r + li) * 64 + ((2 * lg + k) ^ ((li >> 2) & 3)) * 16);
            return mx_v8i{v[0], v[1], v[2], v[3], 0, 0, 0, 0};
        };
        const int left = nb - (4 * i + 2 * lg);
        const uint32_t live = left > 1 ? 0xffffu : left > 0 ? 0xffu : 0u;
        auto scales = [&](int r) { return (int)((*reinterpret_cast<const uint32_t *>(w_scales + (32 * r + li) * 16) >> (16 * lg)) & live); };
        const mx_v8i b00 = codes(0, 0), b01 = codes(0, 1), b10 = codes(1, 0), b11 = codes(1, 1);
        const int scale0 = scales(0), scale1 = scales(1);
        // (macros: as a struct handed between lambdas the operands end up in scratch memory)
        auto piece = [&](int h, int k, int n) { return *reinterpret_cast<const mx_v4i *>(st + h * 32 * MX_ROW + (n >> 1) * 128 + piece_at[k][n & 1]); };
        // step K's operands of half H, requested here, ahead of the products in front of theirs: the planes' dwords 0..3,
        // dwords 4 and 5 of planes 0 and 1, of planes 2 and 3, and the planes' scales
#define FRK_MX_READ(o, H, K)                                                                                           \
    const mx_v4i o##0 = piece(H, K, 0), o##1 = piece(H, K, 1), o##2 = piece(H, K, 2), o##3 = piece(H, K, 3),           \
                 o##01 = piece(H, K, 4), o##23 = piece(H, K, 5);                                                       \
    const int o##_scales = *reinterpret_cast<const int *>(st + MX_STAGE_SCALES + (32 * H + li) * 16 + (2 * lg + K) * 4); \
    __builtin_amdgcn_sched_barrier(0)
#define FRK_MX_PLANE(o, K, P, head, tail, T)                                                                           \
    {                                                                                                                  \
        const mx_v8i x = {head[0], head[1], head[2], head[3], tail[T], tail[T + 1], 0, 0};                             \
        part0 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, b##K##0, part0, E2M3, E2M1, P, o##_scales, K, scale0); \
        part1 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, b##K##1, part1, E2M3, E2M1, P, o##_scales, K, scale1); \
    }
#define FRK_MX_STEP(o, K)                   \
    FRK_MX_PLANE(o, K, 0, o##0, o##01, 0) \
    FRK_MX_PLANE(o, K, 1, o##1, o##01, 2) \
    FRK_MX_PLANE(o, K, 2, o##2, o##23, 0) \
    FRK_MX_PLANE(o, K, 3, o##3, o##23, 2) \
    asm volatile("" : "+v"(part0), "+v"(part1));  // (stays in front of the requests behind it)
        const std::integral_constant<int, 0> c0;
        const std::integral_constant<int, 1> c1;
        const std::integral_constant<int, 2> c2;
        const std::integral_constant<int, 3> c3;
        FRK_MX_READ(p, 0, 0);
        FRK_MX_READ(q, 0, 1);
        request(c0, i);
        mx_v16f part0 = mx_v16f{0.0f}, part1 = part0;
        FRK_MX_STEP(p, 0)
        request(c1, i);
        FRK_MX_READ(u, 1, 0);  // (the stage has the second half's place in any case)
        FRK_MX_STEP(q, 1)
        acc[0][0] += part0;
        acc[0][1] += part1;
        request(c2, i);
        if (two) {
            FRK_MX_READ(v, 1, 1);
            part0 = part1 = mx_v16f{0.0f};
            FRK_MX_STEP(u, 0)
            FRK_MX_STEP(v, 1)
            acc[1][0] += part0;
            acc[1][1] += part1;
        }
        request(c3, i);
#undef FRK_MX_READ
#undef FRK_MX_PLANE
#undef FRK_MX_STEP
    };
    // A quad: its digits and weights have landed (behind them only the digits of quad i + 1 were requested), everybody
    // has left the stage that the next request overwrites.
    for (int c = 0; c < 4; c++) fetch_codes(0, c);
    fetch_weight_scales(0);
    request(std::integral_constant<int, 2>(), -2);
    request(std::integral_constant<int, 3>(), -2);
    request(std::integral_constant<int, 2>(), -1);
    request(std::integral_constant<int, 3>(), -1);
    for (int i = 0; i < quads; i++) {
        if (i + 1 < quads && wave == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(REQUESTS + 1) : "memory");
        else if (i + 1 < quads) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(REQUESTS) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        lds_barrier();
        multiply(i);
    }

    // the factor of row `lane` of the tile
    float factor = 1.0f;
    {
        const int r = tile.y + lane, src = g.src_rows ? g.src_rows[r] : r;
        if (lane < tile.z && src >= 0) factor = g.acts.factor[src];
    }
    const bool scaled_rows = __any(factor != 1.0f);


    // ---- register r of a lane: activation row 8 * (r / 4) + 4 * (lane / 32) + r % 4 of the half, weight row lane % 32
#pragma unroll
    for (int h = 0; h < 2; h++) {
        if (h == 1 && !two) break;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int tok = 32 * h + 8 * (r >> 2) + 4 * lg + (r & 3);
            float v0 = acc[h][0][r], v1 = acc[h][1][r];
            if (scaled_rows) {
                const float f = __shfl(factor, tok);
                v0 = f == 1.0f ? v0 : v0 * f, v1 = f == 1.0f ? v1 : v1 * f;
            }
            if (tok >= tile.z) continue;
            float *dst = g.y + (size_t)(tile.w + tok) * g.rows;
            if (GLU) {
                if (row0 < g.rows) dst[row0] = silu_as_host(v0) * v1;
            } else {
                if (row0 < g.rows) dst[row0] = v0;
                if (row0 + 32 < g.rows) dst[row0 + 32] = v1;
            }
        }
    }
#endif
}

bool mx_gemm_fits(size_t act_rows, size_t rows_g, size_t cols) {
    // lane offsets are 32 bits wide
    return act_rows * mx_padded_blocks(cols) * MX_BLOCK_BYTES <= 0xffffffffu &&
           rows_g * layout_for(FRK_KIND_MXFP4, cols).row_stride <= 0xffffffffu;
}
// up: the second matrix (y = silu(gate) * up), or null
int launch_gemm_mx_grouped(const frk_weights *w, const frk_weights *up, size_t rows_g, const MxActs &acts, const int *src_rows,
                           const int4 *tiles, const int *n_tiles, size_t max_tiles, float *y, hipStream_t s) {
    if (max_tiles == 0) return FRK_OK;
    MxGemmArgs g;
    g.W = w->dev;
    g.W2 = up ? up->dev : nullptr;
    g.row_stride = w->layout.row_stride;
    g.group_stride = rows_g * g.row_stride;
    g.rows = (int)rows_g;
    g.nb = (int)(w->cols / 32);
    g.acts = acts;
    g.src_rows = src_rows;
    g.tiles = tiles;
    g.n_tiles = n_tiles;
    g.y = y;
    const size_t rows_wave = up ? 32 : 64, tiles8 = (max_tiles + 7) / 8 * 8;
    const bool wide = max_tiles * ((rows_g + 8 * rows_wave - 1) / (8 * rows_wave)) >= 256;
    g.row_groups = (int)((rows_g + (wide ? 8 : 4) * rows_wave - 1) / ((wide ? 8 : 4) * rows_wave));
    const size_t grid = tiles8 * (size_t)g.row_groups;
    if (grid > 0x7fffffffu) return set_error(FRK_ERR_SHAPE, "grouped gemm: %zu rows a group, %zu tiles", rows_g, max_tiles);
    static bool sized = false;  // a benign race: every thread sets the same attribute
    if (!sized) {
        const void *k[4] = {reinterpret_cast<const void *>(&gemm_mx_grouped_kernel<8, true>), reinterpret_cast<const void *>(&gemm_mx_grouped_kernel<8, false>),
                            reinterpret_cast<const void *>(&gemm_mx_grouped_kernel<4, true>), reinterpret_cast<const void *>(&gemm_mx_grouped_kernel<4, false>)};
        for (int i = 0; i < 4; i++) {
            const size_t bytes = i < 2 ? mx_lds_bytes<8>() : mx_lds_bytes<4>();
            hipError_t e = hipFuncSetAttribute(k[i], hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
            if (e != hipSuccess) return set_error(FRK_ERR_HIP, "hipFuncSetAttribute(LDS %zu): %s", bytes, hipGetErrorString(e));
        }
        sized = true;
    }
#define FRK_GO(NW, GLU) hipLaunchKernelGGL((gemm_mx_grouped_kernel<NW, GLU>), dim3((unsigned)grid), dim3(64 * NW), mx_lds_bytes<NW>(), s, g)
    if (wide && up) FRK_GO(8, true);
    else if (wide) FRK_GO(8, false);
    else if (up) FRK_GO(4, true);
    else FRK_GO(4, false);
#undef FRK_GO
    FRK_LAUNCH_CHECK("gemm_mx_grouped");
    return FRK_OK;
}

}  // namespace frk
