// Grouped GEMM over MXFP4 experts on the block-scaled matrix cores (v_mfma_scale_f32_32x32x64_f8f6f4):
//   y[token][row] = sum over the 32-wide blocks of  (dw * da) * sum_i qw_i * qa_i
// with the activations quantized to Q8_0 blocks as on every integer path of this kind (dot_mxfp4_q8,
// crates/frink-quant/src/legacy_q8.rs:169-213; the MoE bucket path, crates/frink-models/src/decoder/ffn_batch.rs:343-434).
//
// The matrix core takes an MXFP4 block as it is stored: sixteen bytes of E2M1 codes are a lane's operand, the block's
// E8M0 byte its scale.  The activation block's  da * qa  is a 19-bit number (f16 scale: 11 bits of mantissa, 8-bit quant)
// times a power of two, and goes through as four planes of signed base-32 digits, -16 .. 16: exact in E2M3 (six bits),
// the power of two and the plane's 32^p in its E8M0 scale.  So every product is exact, sums are f32 inside the matrix
// core, and the vector ALU has no float step at all -- it adds the sums of 128 columns onto the running ones.  From 384
// columns on that keeps the error against 64 bits below that of one rounding a block, which shorter rows keep
// (mx_gemm_takes).
// (Byte i of a GGUF block holds elements i and i + 16; a lane's operand takes byte i as k = 2i and 2i + 1.  The order of
// k within a block is free as long as both operands have it: the digits are stored in the weights' order.)
//
// Before, the experts were decoded to signed bytes with f16 scales on every call (83 us a projection of 32 x 2880 x
// 2880) and multiplied by the Q8_0 kernel, whose float step is 32 vector instructions per MFMA (156 us).
#include "frk_mx_quant.hpp"

#include <cmath>
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

MxActs mx_acts_carve(void *base, size_t rows, size_t cols) {
    const size_t blocks = rows * mx_padded_blocks(cols);
    MxActs a;
    a.digits = (uint8_t *)base;
    a.scales = (uint32_t *)((char *)base + round_up(blocks * MX_BLOCK_BYTES, 256));
    a.infinite = (int *)((char *)a.scales + round_up(blocks * 4, 256));
    return a;
}
size_t mx_acts_bytes(size_t rows, size_t cols) {
    const size_t blocks = rows * mx_padded_blocks(cols);
    return round_up(blocks * MX_BLOCK_BYTES, 256) + round_up(blocks * 4, 256) + round_up(rows * 4, 256);
}

// `used`: a row whose entry is negative is left as it is
// A block of the row a quad of lanes, all of them at once: with 128 threads a row its blocks were three trips to memory one
// after the other (2048 rows of 2880 columns are bound by the vector ALU either way; with the token rows'
// digits likewise, 32 experts top-4 of 2880 / 2880 at 64 tokens, the layer, 184 -> 175 us, 16 experts at 24 117 -> 110.5).
__global__ __launch_bounds__(512) void quantize_mx_kernel(const float *__restrict__ x, int nb, const int *__restrict__ used, MxActs out) {
    __shared__ int infinite;
    const int row = blockIdx.x;
    if (used && used[row] < 0) return;
    if (threadIdx.x == 0) infinite = 0;
    __syncthreads();
    quantize_mx_row(x, row, nb, threadIdx.x, (int)blockDim.x, &infinite, out);
}
int launch_quantize_mx(const float *x, size_t rows, size_t cols, const int *used, const MxActs &out, hipStream_t s) {
    if (rows == 0) return FRK_OK;
    const unsigned threads = (unsigned)std::min<size_t>((4 * mx_padded_blocks(cols) + 63) / 64 * 64, 512);
    hipLaunchKernelGGL(quantize_mx_kernel, dim3((unsigned)rows), dim3(threads), 0, s, x, (int)(cols / 32), used, out);
    FRK_LAUNCH_CHECK("quantize_mx");
    return FRK_OK;
}

// ---- the GEMM.  A workgroup of NW wavefronts multiplies one tile (at most 96 activation rows of one group, halves
// of 32) with 64 weight rows a wavefront, as two groups of 32: of one matrix, or (GLU) the same rows of gate and up,
// whose results meet in the epilogue as silu(gate) * up.
//
// The columns go by four blocks at a time: step s (0, 1) multiplies blocks s and 2 + s, a lane block s or 2 + s of its
// row by its half (k = 64).  Everything comes straight into LDS: the activations' digits (37 KB) into two stages that the
// workgroup shares, a quad refilled as soon as everybody has read it, with one barrier a quad; the weights two quads of
// blocks ahead into a wavefront's own two slots, their scale bytes four quads at a time.
// A quad of a full tile takes about 2.9 us: 96 products a SIMD at the 22 ns that a chain of E2M3 x E2M1 products alone was
// measured at (the chip holds 1.6 GHz under it) are 2.1; without its requests 2.5.  So neighbouring lanes of a request
// fetch neighbouring pieces of memory (384 bytes of digits, 64 of codes a row), the LDS images are swizzled so that a
// fragment's reads -- one piece of sixteen rows each -- fall in different banks, and the requests are spread over the
// arithmetic.  Gate and up of 32 experts of 2880 x 2880 over 2048 pairs: weights loaded into registers, a row a lane, 227
// us; weights in LDS but a lane per activation row 208; every request at the head of its quad 181; operands of the next
// quad read behind the barrier instead of in front of the last step 171; tiles of 64 rows 152-159; tiles of 96 rows (half of
// the experts have more than 64 pairs and read their weights a second time for a few rows otherwise) 145, with silu ahead of
// the stores 142, an XCD's last jobs cut in two 132; the down projection 90 -> 72 (the bytes from memory take 50 and 27).
// A step's operands are read in two parts of twelve registers, as three halves' sums leave no room for a second step's.
// Eight wavefronts a workgroup where that still fills the chip: a stage of digits then serves twice the rows (the down
// projection 137 -> 97 us). ----
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
constexpr int MX_STAGE_SCALES = MX_TILE * MX_ROW;      // [MX_TILE rows][4 blocks] dwords
constexpr int MX_STAGE = MX_STAGE_SCALES + MX_TILE * 16;
constexpr int MX_STAGES = 2;
constexpr int XCD_CUS = 32;
static_assert(MX_TILE == 96, "three halves");
constexpr int MX_W_SCALES = 2 * 4096;                  // two slots of codes [64 rows][4 blocks], two of scales [64 rows][16]
constexpr int MX_W_WAVE = MX_W_SCALES + 2 * 1024;
template <int NW>
constexpr size_t mx_lds_bytes() { return (size_t)MX_STAGES * MX_STAGE + (size_t)NW * MX_W_WAVE + sizeof(EXPF_TABLE); }
static_assert(mx_lds_bytes<8>() <= 160 * 1024, "LDS of a CU");

template <int NW, bool GLU>
__global__ __launch_bounds__(64 * NW, 2) void gemm_mx_grouped_kernel(MxGemmArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
    extern __shared__ __align__(16) uint8_t mx_lds[];
    uint8_t *const lds = mx_lds;
    // The workgroups of a tile sit on one XCD (block id mod 8), whose L2 then serves the tile's digits.  One workgroup fits a
    // CU, so an XCD's jobs go in rounds of 32; where the last round is half empty, its jobs are cut in two: half the
    // rows each, four wavefronts to multiply them and the other four to help with the digits' requests.
    const int xcd = (int)blockIdx.x & 7, jobs = max(*g.n_tiles - xcd + 7, 0) / 8 * g.row_groups;
    int j = (int)blockIdx.x >> 3, part = -1;
    if (NW == 8) {
        const int last = jobs % XCD_CUS;
        if (last <= XCD_CUS / 2 && j >= jobs - last) {
            part = (j - (jobs - last)) & 1;
            j = jobs - last + ((j - (jobs - last)) >> 1);
        }
    }
    if (j >= jobs) return;
    const int t = xcd + 8 * (j / g.row_groups);
    const int4 tile = g.tiles[t];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int li = lane & 31, lg = lane >> 5;
    const int nb = g.nb, nbp = (nb + 7) & ~7;
    const int quads = (nb + 3) >> 2;
    uint64_t *const expf_table = reinterpret_cast<uint64_t *>(lds + MX_STAGES * MX_STAGE + NW * MX_W_WAVE);
    if (GLU && threadIdx.x < 32) expf_table[threadIdx.x] = EXPF_TABLE[threadIdx.x];  // (read behind the first barrier)
    const int halves = (tile.z + 31) >> 5;  // of 32 rows, three at most

    const uint32_t lds0 = lds_address(lds);
    // ---- weights: rows row0 + lane % 32 of the two groups.  Request c of a quad brings rows 16c .. 16c + 15 of the 64:
    // slot p of row r holds block p ^ (r / 4) % 4, so that the reads of one block of 32 rows fall in different banks.
    const int row_wave = ((j % g.row_groups) * NW + (part < 0 ? wave : part * 4 + (wave & 3))) * (GLU ? 32 : 64), row0 = row_wave + li;
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

    // ---- activations: a stage's digits are rows of 24 pieces, piece s of row r in place s ^ (r / 2) % 8 (sixteen rows reading one
    // piece each then touch sixteen different pieces of the 64 banks).  A half is twelve requests, dealt out to the wavefronts;
    // the first two fetch the scales.
    constexpr int REQUESTS = 36 / NW + (36 % NW != 0);
    auto act_row = [&](int r) { return (uint32_t)(g.src_rows ? max(g.src_rows[tile.y + r], 0) : tile.y + r); };
    uint32_t digits_off[REQUESTS];
#pragma unroll
    for (int c = 0; c < REQUESTS; c++) {
        const int at = min(wave + c * NW, 12 * halves - 1) * 64 + lane, r = at / 24;
        digits_off[c] = act_row(r) * (uint32_t)nbp * MX_BLOCK_BYTES + (uint32_t)((at % 24) ^ ((r >> 1) & 7)) * 16;
    }
    const int scales_row = (wave & 1) * 64 + lane;
    const bool fetches_scales = wave < 2 && scales_row < 32 * halves;
    const uint32_t scales_off = fetches_scales ? act_row(scales_row) * (uint32_t)nbp * 4 : 0u;
    auto request_digits = [&](int i) {  // of quad i + 2, when everybody has read quad i's
        if (i + 2 >= quads) return;
        const uint32_t to = lds0 + (uint32_t)(i & 1) * MX_STAGE;
#pragma unroll
        for (int c = 0; c < REQUESTS; c++)
            if (wave + c * NW < 12 * halves)
                dma16(to + (uint32_t)(wave + c * NW) * 1024, g.acts.digits + (size_t)(i + 2) * MX_ROW, digits_off[c]);
        if (fetches_scales) dma16(to + MX_STAGE_SCALES + (uint32_t)(wave & 1) * 1024, g.acts.scales + (size_t)(i + 2) * 4, scales_off);
    };
    // the codes of quad i + 2, whose slot is that of quad i, in the wavefront's registers by then; spread over the arithmetic (all at once, the
    // requests of eight wavefronts hold each other up)
    auto request_codes = [&](int i, int c) {
        if (i + 2 >= quads) return;
        fetch_codes(i + 2, c);
        fetch_codes(i + 2, c + 1);
        if (c == 0 && ((i + 2) & 3) == 0) fetch_weight_scales(i + 2);
    };
    // where this lane's pieces of step k sit in a half's 32 rows: piece 4n + block in place (4n + block) ^ x, so the even n
    // 128 bytes apart from here, the odd ones from there
    uint32_t piece_at[2][2];
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int n = 0; n < 2; n++) piece_at[k][n] = (uint32_t)(li * MX_ROW + ((4 * n + 2 * lg + k) ^ ((li >> 1) & 7)) * 16);

    mx_v16f acc[3][2];  // [half][row group]
#pragma unroll
    for (int h = 0; h < 3; h++)
#pragma unroll
        for (int r = 0; r < 2; r++) acc[h][r] = mx_v16f{0.0f};

    // One quad: per half two steps of four planes of digits, smallest first, their sum added onto the running one.  Operands
    // are read while others are multiplied -- across the quads too: before the last step's second part the next quad is
    // waited for (and everybody has read the present one), and its codes and first operands are read behind that part's
    // products.
    // (macros: as a struct handed between lambdas the operands end up in scratch memory)
    constexpr int E2M3 = 2, E2M1 = 4;
    const uint8_t *const w_wave = lds + MX_STAGES * MX_STAGE + (size_t)wave * MX_W_WAVE;
    auto codes = [&](int i, int k, int r) {  // of step k and row group r
        return *reinterpret_cast<const mx_v4i *>(w_wave + (i & 1) * 4096 + (32 * r + li) * 64 + ((2 * lg + k) ^ ((li >> 2) & 3)) * 16);
    };
    auto scales = [&](int i, int r) {  // the scale bytes of the lane's two blocks (a block past the row's end: 2^-127)
        const int left = nb - (4 * i + 2 * lg);
        const uint32_t live = left > 1 ? 0xffffu : left > 0 ? 0xffu : 0u;
        const uint32_t four = *reinterpret_cast<const uint32_t *>(w_wave + MX_W_SCALES + ((i >> 2) & 1) * 1024 + (i & 3) * 4 + (32 * r + li) * 16);
        return (int)((four >> (16 * lg)) & live);
    };
    auto piece = [&](const uint8_t *st, int h, int k, int n) {
        return *reinterpret_cast<const mx_v4i *>(st + h * 32 * MX_ROW + (n >> 1) * 128 + piece_at[k][n & 1]);
    };
    auto act_scales = [&](const uint8_t *st, int h, int k) {
        return *reinterpret_cast<const int *>(st + MX_STAGE_SCALES + (32 * h + li) * 16 + (2 * lg + k) * 4);
    };
    // A step's operands come in two parts, planes 0 and 1 (A: dwords 0..3 of each, then dwords 4 and 5 of both; with the
    // planes' scales) and planes 2 and 3 (B): one is read while the other is multiplied.
#define FRK_MX_READ_A(H, K)                                                                                            \
    a0 = piece(st, H, K, 0), a1 = piece(st, H, K, 1), a01 = piece(st, H, K, 4), next_scales = act_scales(st, H, K);    \
    __builtin_amdgcn_sched_barrier(0)
#define FRK_MX_READ_B(H, K)                                                                                            \
    b2 = piece(st, H, K, 2), b3 = piece(st, H, K, 3), b23 = piece(st, H, K, 5);                                        \
    __builtin_amdgcn_sched_barrier(0)
#define FRK_MX_PLANE(K, P, head, tail, T)                                                                              \
    {                                                                                                                  \
        const mx_v8i x = {head[0], head[1], head[2], head[3], tail[T], tail[T + 1], 0, 0};                             \
        const mx_v8i y0 = {w##K##0[0], w##K##0[1], w##K##0[2], w##K##0[3], 0, 0, 0, 0};                                \
        const mx_v8i y1 = {w##K##1[0], w##K##1[1], w##K##1[2], w##K##1[3], 0, 0, 0, 0};                                \
        part0 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, y0, part0, E2M3, E2M1, P, act_scale, K, scale0);    \
        part1 = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(x, y1, part1, E2M3, E2M1, P, act_scale, K, scale1);    \
    }
#define FRK_MX_MULTIPLY_A(K)                          \
    act_scale = next_scales;                          \
    FRK_MX_PLANE(K, 0, a0, a01, 0)                    \
    FRK_MX_PLANE(K, 1, a1, a01, 2)                    \
    asm volatile("" : "+v"(part0), "+v"(part1));
#define FRK_MX_MULTIPLY_B(K)                          \
    FRK_MX_PLANE(K, 2, b2, b23, 0)                    \
    FRK_MX_PLANE(K, 3, b3, b23, 2)                    \
    asm volatile("" : "+v"(part0), "+v"(part1));  // (stays in front of the requests behind it)
    // quad I has landed: behind its digits the wavefront requested the codes of quad I + 1 (four times, and now and then
    // scales: then a little more is waited for); afterwards its codes (step 0's in place, step 1's beside the present ones)
    // and first operands
#define FRK_MX_ARRIVE(I)                                                                                               \
    if ((I) + 1 < quads) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");                                              \
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                                                              \
    lds_barrier();                                                                                                     \
    st = lds + (size_t)((I) & 1) * MX_STAGE;                                                                           \
    w00 = codes(I, 0, 0), w01 = codes(I, 0, 1);                                                                    \
    next_scale0 = scales(I, 0), next_scale1 = scales(I, 1);                                                            \
    __builtin_amdgcn_sched_barrier(0);                                                                                 \
    FRK_MX_READ_A(0, 0)
    auto all_quads = [&](auto halves_c) {
        constexpr int H = decltype(halves_c)::value;
        const uint8_t *st;
        mx_v4i w00, w01, w10, w11, a0, a1, a01, b2, b3, b23;
        int scale0, scale1, next_scale0, next_scale1, act_scale, next_scales;
        FRK_MX_ARRIVE(0);
        request_digits(-1);
        scale0 = next_scale0, scale1 = next_scale1;
        for (int i = 0; i < quads; i++) {
#pragma unroll
            for (int h = 0; h < H; h++) {
                mx_v16f part0 = mx_v16f{0.0f}, part1 = part0;
                FRK_MX_READ_B(h, 0);
                FRK_MX_MULTIPLY_A(0)
                if (h == 0) w10 = codes(i, 1, 0), w11 = codes(i, 1, 1);
                FRK_MX_READ_A(h, 1);
                FRK_MX_MULTIPLY_B(0)
                FRK_MX_READ_B(h, 1);
                FRK_MX_MULTIPLY_A(1)
                if (h == 0) request_codes(i, 0);
                if (H == 1) request_codes(i, 2);
                if (h < H - 1) {
                    FRK_MX_READ_A(h + 1, 0);
                } else {
                    FRK_MX_ARRIVE(i + 1);  // (behind the last quad: whatever lies there, unused)
                    request_digits(i);
                }
                FRK_MX_MULTIPLY_B(1)
                acc[h][0] += part0;
                acc[h][1] += part1;
                if (H == 3) asm volatile("" : "+v"(acc[h][0]), "+v"(acc[h][1]));  // (sunk further down, two halves' sums are alive at once)
                if (h == 0 && H > 1) request_codes(i, 2);
            }
            scale0 = next_scale0, scale1 = next_scale1;
        }
    };
    request_digits(-2);
    if (part >= 0 && wave >= 4) {  // a helper: the same barriers
        for (int i = -1; i < quads; i++) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            lds_barrier();
            request_digits(i);
        }
        return;
    }
    for (int c = 0; c < 4; c++) fetch_codes(0, c);
    fetch_weight_scales(0);
    request_codes(-1, 0);
    request_codes(-1, 2);
    if (halves > 2) all_quads(std::integral_constant<int, 3>());
    else if (halves > 1) all_quads(std::integral_constant<int, 2>());
    else all_quads(std::integral_constant<int, 1>());
#undef FRK_MX_READ_A
#undef FRK_MX_READ_B
#undef FRK_MX_PLANE
#undef FRK_MX_MULTIPLY_A
#undef FRK_MX_MULTIPLY_B
#undef FRK_MX_ARRIVE

    // ---- register r of a lane: activation row 8 * (r / 4) + 4 * (lane / 32) + r % 4 of the half, weight row lane % 32
    // (silu ahead of the stores and their conditions, so that several values' chains of operations run beside each other)
#pragma unroll
    for (int h = 0; h < 3; h++) {
        if (h >= halves) break;
        if (GLU) {
#pragma unroll
            for (int r = 0; r < 16; r++) acc[h][0][r] = silu_as_host(acc[h][0][r], expf_table) * acc[h][1][r];
        }
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int tok = 32 * h + 8 * (r >> 2) + 4 * lg + (r & 3);
            if (tok >= tile.z) continue;
            float *dst = g.y + (size_t)(tile.w + tok) * g.rows;
            if (row0 < g.rows) dst[row0] = acc[h][0][r];
            if (!GLU && row0 + 32 < g.rows) dst[row0 + 32] = acc[h][1][r];
        }
    }

    // ---- the rows with infinite blocks again (hardly ever any): what decides is the sign of each such block's integer
    // sum, an infinity each, NaN where the sum is zero or two differ.  Lanes 0 .. 31 take the first row group, the others
    // the second.
    auto infinite_rows = [&](int first) {  // of 64 rows
        bool again = false;
        if (first + lane < tile.z) {
            const int src = g.src_rows ? g.src_rows[tile.y + first + lane] : tile.y + first + lane;
            again = src >= 0 && g.acts.infinite[src] != 0;
        }
        return __ballot(again);
    };
    uint64_t left = infinite_rows(0), left_high = tile.z > 64 ? infinite_rows(64) : 0;
    if (left | left_high) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (their first results are out)
    while (left | left_high) {
        const int tok = left ? __builtin_ctzll(left) : 64 + __builtin_ctzll(left_high);
        if (left) left &= left - 1;
        else left_high &= left_high - 1;
        const size_t first = (size_t)act_row(tok) * nbp;
        const uint8_t *codes_row = (lg ? w_base[1] : w_base[0]) + weight_row(lane);
        float sum = 0.0f;
        for (int b = 0; b < nb; b++) {
            if ((g.acts.scales[first + b] & 0xffu) != MX_INFINITE) continue;
            const int8_t *q = reinterpret_cast<const int8_t *>(g.acts.digits + (first + b) * MX_BLOCK_BYTES);
            int isum = 0;
            for (int i = 0; i < 16; i++) {
                auto times = [&](int code, int quant) {  // 0, 1, 2, 3, 4, 6, 8, 12 halves
                    const int m = (int)(0xc8643210u >> (4 * (code & 7)) & 15u);
                    return (code & 8 ? -m : m) * quant;
                };
                isum += times(codes_row[b * 16 + i] & 15, q[i]) + times(codes_row[b * 16 + i] >> 4, q[16 + i]);
            }
            sum += (float)isum * __builtin_inff();
        }
        float *dst = g.y + (size_t)(tile.w + tok) * g.rows;
        if (GLU) {
            const float up = __shfl_xor(sum, 32);
            if (lg == 0 && row0 < g.rows) dst[row0] = silu_as_host(sum, expf_table) * up;
        } else if (row0 + 32 * lg < g.rows) {
            dst[row0 + 32 * lg] = sum;
        }
    }
#endif
}

// Rows of 384 columns and more.  A matrix-core step rounds its 64 products several times within the last places of the
// largest, and the vector ALU adds once a quad of blocks; the decoded form's kernel rounds once a block.  Errors against
// 64-bit sums of the same quantized operands, this kernel's over the other one's (2-norm / largest; activations N(0, 1) with
// scales of 4 powers of two, and the worst of that, of scales of 40 powers and of a 64th of the channels fifty times as
// large): 64 columns 1.02 / 1.00 and 1.30 / 1.54, 128 1.01 / 0.94 and 1.25 / 1.52, 256 0.90 / 0.73 and 1.08 / 0.93, 320 0.91 /
// 0.83 and 1.03 / 0.86, 384 0.85 / 0.71 and 0.99 / 0.84, 512 0.83 / 0.68 and 0.94 / 0.85, 1024 0.76 / 0.67 and 0.83 / 0.81, 2880
// 0.68 / 0.51 and 0.76 / 0.56 (there 9.3e-8 against 1.4e-7 in the 2-norm).
bool mx_gemm_takes(size_t act_rows, size_t rows_g, size_t cols) {
    if (cols < 384) return false;
    // lane offsets are 32 bits wide
    return act_rows * mx_padded_blocks(cols) * MX_BLOCK_BYTES <= 0xffffffffu &&
           rows_g * layout_for(FRK_KIND_MXFP4, cols).row_stride <= 0xffffffffu;
}
// Wavefronts of a workgroup: eight where 64-row tiles of as many groups as may be partly used fill the chip.
static int mx_waves(size_t pairs, size_t groups, size_t rows_g, bool glu) {
    const size_t rows = 8 * (glu ? 32 : 64);
    return (pairs / 64 + groups) * ((rows_g + rows - 1) / rows) >= 256 ? 8 : 4;
}
// Tiles of so many rows that pairs dealt to the groups at random take: a group's number is about normal around the mean.
static double expected_tiles(size_t pairs, size_t groups, double rows) {
    const double mean = (double)pairs / (double)groups, spread = std::sqrt(2.0 * mean);
    const double sure = std::max(0.0, std::floor((mean - 3.0 * spread) / rows));  // every group has these
    double tiles = sure, p = 1.0;
    for (double j = sure; p > 1e-3; j++) tiles += p = 0.5 * std::erfc((j * rows + 0.5 - mean) / spread);  // more than j * rows
    return tiles * (double)groups;
}
// Tiles of 96 rows where the workgroups of 64-row tiles would not fit the chip's 256 CUs at once (with 1 % on top: the numbers
// differ): an expert of 65 to 96 pairs then reads its weights once, not a second time for a few rows.  Tiles of 64 rows where they do:
// there a job's length is the launch's.  As eight wavefronts a workgroup take over from four with more pairs (mx_waves), the
// workgroups become half as many and fit again.  Measured in us a layer, 64-row tiles / 96: where they do not fit, 32 experts
// top-4 of 2880 / 2880 at 517 tokens 242 / 212, 16 top-2 of 2240 / 1312 at 741 106 / 88, 8 top-2 of 2880 / 2880 at 768 182 / 152; where they just
// fit, of four wavefronts, 8 top-2 of 2048 / 2048 at 416 72 / 87, of eight, 8 top-2 of 2880 / 2880 at 448 108 / 122, 16 top-2 of 1536 / 1536 at
// 864 77 / 86.  Nor where four wavefronts' workgroups, whose jobs are not cut in two, need two rounds with either tile: 8
// top-4 of 2304 / 1088 at 694 tokens 124 / 148.  Over 278 drawn layers the choice is 0.8 % behind the better one on average, 12 % at
// most; none is slower than before there were tiles of 96 rows.
int mx_tile(size_t pairs, size_t groups, size_t rows_g, bool glu) {
    const int waves = mx_waves(pairs, groups, rows_g, glu);
    const size_t rows = (size_t)waves * (glu ? 32 : 64);
    const double row_groups = (double)((rows_g + rows - 1) / rows), round = 1.01 * 256.0;
    const double of64 = expected_tiles(pairs, groups, MOE_TILE) * row_groups;
    if (of64 <= round) return MOE_TILE;
    if (waves == 4 && of64 <= 512.0 && expected_tiles(pairs, groups, MX_TILE) * row_groups > round) return MOE_TILE;
    return MX_TILE;
}
// up: the second matrix (y = silu(gate) * up), or null
int launch_gemm_mx_grouped(const frk_weights *w, const frk_weights *up, size_t rows_g, const MxActs &acts, const int *src_rows,
                           const int4 *tiles, const int *n_tiles, size_t max_tiles, size_t pairs, size_t groups, float *y, hipStream_t s) {
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
    const bool wide = mx_waves(pairs, groups, rows_g, up != nullptr) == 8;
    g.row_groups = (int)((rows_g + (wide ? 8 : 4) * rows_wave - 1) / ((wide ? 8 : 4) * rows_wave));
    const size_t grid = tiles8 * (size_t)g.row_groups + (wide ? 8 * XCD_CUS / 2 : 0);
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
