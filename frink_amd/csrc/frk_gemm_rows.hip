// Batches of 2 to 32 rows of the K-quants on the matrix cores (batched decoding), and larger ones of small matrices, every 32 tokens by
// workgroups of their own (blockIdx.y): y[tok][row] is dot_q{4,5,6}_k_q8's
// (crates/frink-quant/src/lib.rs:822-869, 886-938, 1069-1110), the integers exact, the float step the thin kernels'.
//
// A workgroup is sixteen weight rows, its wavefronts shares of the columns.  A wavefront streams its share two blocks at a
// time into an LDS slot of its own (global_load_lds) and multiplies them against the batch's tiles, whose operands come from
// L2 straight into registers, a kilobyte a load, in the order in which the matrix core wants them.  Nothing is shared
// before the sums: no barrier stands between requests and arithmetic, and the wavefronts' sums are added once, in pairs.
//
// What it replaces: the thin kernels stage a batch's quants in LDS (up to 8 or 16 rows of it, a second round or launch behind
// them), and the 64 x 32 tiles of the pipelined GEMM leave most of the chip idle below 14000 rows or split a row's blocks
// between workgroups, with a launch to add their sums.
#include "frk_gemm_pipe.hpp"

namespace frk {

typedef _Float16 v4h __attribute__((ext_vector_type(4)));

struct RowsArgs {
    const uint8_t *W;
    size_t row_stride;
    uint32_t off_qh, off_sc, off_d;  // the planes of a Q6_K row
    int rows, nb, M;
    int each;     // pairs of blocks of a wavefront
    Q8KTiled a;   // one tile of 32 tokens, or
    Q8KActs plain;
    float *y;     // [M][rows]
};
constexpr int ROWS_WAVES = 8;

#if defined(__HIP_DEVICE_COMPILE__)
// The activations behind buffer descriptors: a load's address is a lane offset and a scalar one.  As plain rows, not
// tiles, a load touches a line for every token (Q4_K and Q5_K: the quants come through LDS, see stage).
template <bool PLAIN>
struct RowsActs {
    __amdgpu_buffer_rsrc_t q, sums, d;
    int nb, M;
    __device__ __forceinline__ v4f scales(int kb, int t, int g) const {  // of tokens 16t + 4g .. + 3
        if constexpr (PLAIN) {
            v4f o;
#pragma unroll
            for (int r = 0; r < 4; r++) o[r] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(d, min(16 * t + 4 * g + r, M - 1) * nb * 4, kb * 4, 0));
            return o;
        }
        return __builtin_bit_cast(v4f, __builtin_amdgcn_raw_buffer_load_b128(d, 16 * g, kb * 128 + 64 * t, 0));
    }
};

// How sixteen weight rows of two blocks come into LDS, leave it for registers and are multiplied: lane (row, g) of the
// sixteen rows and four groups of k.
//
// Q4_K, Q5_K: a row's sixteen-byte pieces back to back and one more, an odd number (a read of sixteen rows then falls in
// different banks), piece 64c + lane in request c.  (What the second block of a last, odd one and the odd piece hold is
// not used; a resident copy ends in 256 bytes of slack.)  A sub-block is one 16x16x32 product, its scale multiplies the four
// results a lane has of its own row: half the vector instructions that two pre-scaled planes take for one tile of tokens
// of Q5_K, a quarter less for Q4_K.
template <int KIND>
struct RowsSide {
    static constexpr bool Q5 = KIND == FRK_KIND_Q5_K;
    static constexpr int BB = Q5 ? Q5_K_BYTES : Q4_K_BYTES, PR = 2 * BB / 16 + 1, ROW = PR * 16, SLOT = 16 * ROW;
    static constexpr int NC = (16 * PR + 63) / 64;
    static_assert(PR % 2 == 1 && 16 * PR <= 64 * NC, "an odd number of pieces a row");
    uint32_t row_at, eight_at;
    int last;
    __device__ __forceinline__ RowsSide(const RowsArgs &, int lane, int last_row) {
        row_at = (uint32_t)((lane & 15) * ROW);
        eight_at = row_at + (uint32_t)(lane >> 4) * 8;
        last = last_row;
    }
    __device__ __forceinline__ void fetch(const RowsArgs &g, uint32_t slot, const uint8_t *first, int kb, int lane) const {
        const uint8_t *from = first + (size_t)kb * BB;
        const uint32_t stride = (uint32_t)g.row_stride;
        asm volatile("" : "+v"(lane));  // (the offsets are made again for each pair, not held in registers)
        uint32_t r = (uint32_t)lane / PR, q = (uint32_t)lane % PR;
#pragma unroll
        for (int c = 0; c < NC; c++) {  // (rows past the matrix repeat the last one)
            if (64 * c + 63 < 16 * PR || 64 * c + lane < 16 * PR) dma16(slot + c * 1024, from, min(r, (uint32_t)last) * stride + q * 16);
            r += 64 / PR, q += 64 % PR;
            if (q >= (uint32_t)PR) q -= PR, r++;
        }
    }
    struct Raw {
        v4i wh;
        v2i q[4], fh;
    };
    __device__ __forceinline__ void read(Raw &R, const uint8_t *slot, int b, int, int) const {
        R.wh = *reinterpret_cast<const v4i *>(slot + row_at + b * BB);
        const uint8_t *eight = slot + eight_at + b * BB;
        if (Q5) R.fh = *reinterpret_cast<const v2i *>(eight + 16);
#pragma unroll
        for (int c = 0; c < 4; c++) R.q[c] = *reinterpret_cast<const v2i *>(eight + (Q5 ? 48 : 16) + 32 * c);
    }
    static __device__ __forceinline__ void arrived(Raw &R) {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(R.wh), "+v"(R.q[0]), "+v"(R.q[1]), "+v"(R.q[2]), "+v"(R.q[3])::"memory");
        if (Q5) asm volatile("" : "+v"(R.fh));
    }
    struct Acts {  // sixteen tokens of a block: lane (token, g)
        v2i q[8];  // 32s + 8g .. + 7
        v4h sums;  // of the groups of sixteen 4g .. 4g + 3
        v4f d;     // of tokens 4g .. 4g + 3
    };
    static __device__ __forceinline__ void load_acts(Acts &A, const RowsActs<false> &a, int kb, int t, int tok, int g) {
        const int at = (g >> 1) * 512 + tok * 16 + (g & 1) * 8;
#pragma unroll
        for (int s = 0; s < 8; s++) A.q[s] = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(a.q, at, kb * 8192 + 1024 * s, 0));
        A.sums = __builtin_bit_cast(v4h, __builtin_amdgcn_raw_buffer_load_b64(a.sums, at, kb * 1024, 0));
        A.d = a.scales(kb, t, g);
    }
    // Of plain rows a load of eight bytes a lane touches a line for every token, twice.  So their quants come through LDS, sixteen tokens
    // of a block as four requests of whole rows' 256 bytes, piece p of token t in place p ^ t (a read's sixteen tokens then fall in different
    // banks), and the next block's are asked for in front of the products and not behind them: 16 tokens of 525 x 4096 in Q4_K 6.7 -> 4.1 us, 3 of
    // 2132 x 13056 in Q5_K 14.0 -> 10.8 (the thin kernels: 4.7 and 12.6).
    struct Small {  // a block's sums as they are, and its scales
        v2i sums;
        v4f d;
    };
    static __device__ __forceinline__ void stage(uint32_t lds, const int8_t *q, const uint32_t (&from)[4], int kb) {
#pragma unroll
        for (int c = 0; c < 4; c++) dma16(lds + c * 1024, q + (size_t)kb * QK_K, from[c]);
    }
    static __device__ __forceinline__ void load_small(Small &S, const RowsActs<true> &a, int kb, int tok, int g) {
        S.sums = __builtin_bit_cast(v2i, __builtin_amdgcn_raw_buffer_load_b64(a.sums, tok * a.nb * 32 + 8 * g, kb * 32, 0));
        S.d = a.scales(kb, 0, g);
    }
    static __device__ __forceinline__ void take(Acts &A, const Small &S, const uint8_t *staged, int lane) {
        const int tok = lane & 15, g = lane >> 4;
        const uint8_t *const mine = staged + tok * QK_K + (g & 1) * 8;
        const int place = (tok ^ (g >> 1)) << 4;
#pragma unroll
        for (int s = 0; s < 8; s++) A.q[s] = *reinterpret_cast<const v2i *>(mine + (place ^ (s << 5)));
        A.sums = v4h{(_Float16)(short)S.sums.x, (_Float16)(short)(S.sums.x >> 16), (_Float16)(short)S.sums.y, (_Float16)(short)(S.sums.y >> 16)};
        A.d = S.d;
#pragma unroll
        for (int s = 0; s < 8; s++) asm volatile("" : "+v"(A.q[s]));
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    }
    // sum[t][r] += weight row lane % 16 times token 16t + 4g + r
    template <int TT>
    static __device__ __forceinline__ void multiply(const Raw &R, int g, const Acts (&A)[TT], v4f (&sum)[TT]) {
        const BlockScales S = block_scales(R.wh);
        v4i s1[TT];
#pragma unroll
        for (int s = 0; s < 8; s++) {
            v2i w;
#pragma unroll
            for (int c = 0; c < 2; c++) {
                uint32_t codes = ((uint32_t)R.q[s >> 1][c] >> (s & 1 ? 4 : 0)) & 0x0f0f0f0fu;
                if (Q5) codes |= (s < 5 ? (uint32_t)R.fh[c] << (4 - s) : (uint32_t)R.fh[c] >> (s - 4)) & 0x10101010u;
                w[c] = (int)codes;
            }
            const int sc = (int)((s < 4 ? S.sc_lo : S.sc_hi) >> (8 * (s & 3)) & 0xffu);
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const v4i dot = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, A[t].q[s]), __builtin_bit_cast(long, w), v4i{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 4; r++) s1[t][r] = s ? s1[t][r] + __mul24(dot[r], sc) : __mul24(dot[r], sc);
            }
            // (two tiles: the products of all eight sub-blocks at once take the registers of a second workgroup)
            if (TT == 2 && (s & 1)) asm volatile("" : "+v"(s1[0]), "+v"(s1[TT - 1]));
        }
        const uint32_t mw = (g & 2 ? S.m_hi : S.m_lo) >> (16 * (g & 1));
        const _Float16 m0 = (_Float16)(int)(mw & 0xff), m1 = (_Float16)(int)((mw >> 8) & 0xff);
        const float d = h2f((uint32_t)R.wh.x & 0xffffu), ndmin = -h2f((uint32_t)R.wh.x >> 16);
#pragma unroll
        for (int t = 0; t < TT; t++) {
            const v4f s2 = __builtin_amdgcn_mfma_f32_16x16x16f16(A[t].sums, v4h{m0, m0, m1, m1}, v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) sum[t][r] = fmaf(A[t].d[r], fmaf(ndmin, s2[r], d * (float)s1[t][r]), sum[t][r]);
        }
    }
};
// Q6_K: lines of 128 bytes (a block's ql; two blocks' qh), eight rows a request, piece p of row r in place p ^ (r / 2) % 8; one more
// request for the scales and the sixteen bytes around the blocks' d.  Two int8 planes (byte_planes): lane (row, g) holds
// weights 64j + 16g .. + 15, one group, of operand j.
template <>
struct RowsSide<FRK_KIND_Q6_K> {
    static constexpr int QH = 4096, SC = 6144, D = SC + 512, SLOT = D + 256;
    uint32_t line[2], small, step, ql_at, qh_at, sc_at;
    __device__ __forceinline__ RowsSide(const RowsArgs &g, int lane, int last_row) {
        const uint32_t stride = (uint32_t)g.row_stride;
#pragma unroll
        for (int h = 0; h < 2; h++) {
            const int r = 8 * h + (lane >> 3);
            line[h] = (uint32_t)min(r, last_row) * stride + (uint32_t)((lane & 7) ^ ((r >> 1) & 7)) * 16;
        }
        const bool is_sc = lane < 32;  // two lanes a row, sixteen lanes for d
        const int r = is_sc ? lane >> 1 : lane & 15;
        small = (uint32_t)min(r, last_row) * stride + (is_sc ? g.off_sc + (uint32_t)((lane & 1) ^ (r >> 3)) * 16 : g.off_d);
        step = is_sc ? 16 : 2;
        const uint32_t lr = (uint32_t)lane & 15, lq = (uint32_t)lane >> 4, x = lr >> 1;
        const uint32_t at = (lr >> 3) * 1024 + (lr & 7) * 128;
        ql_at = at + ((lq ^ x) << 4);        // piece 4n + g, bit 6 turned over for n = 1
        qh_at = at + (((lq & 1) ^ x) << 4);  // piece 4b + 2n + g % 2 likewise
        sc_at = lr * 32 + ((lr >> 3) << 4);  // block b: bit 4 turned over for b = 1
    }
    __device__ __forceinline__ void fetch(const RowsArgs &g, uint32_t slot, const uint8_t *first, int kb, int lane) const {
#pragma unroll
        for (int c = 0; c < 4; c++) dma16(slot + c * 1024, first + (size_t)(kb + (c >> 1)) * 128, line[c & 1]);
#pragma unroll
        for (int c = 0; c < 2; c++) dma16(slot + QH + c * 1024, first + g.off_qh + (size_t)kb * 64, line[c]);
        if (lane < 48) dma16(slot + SC, first, (small + (uint32_t)kb * step) & ~15u);
    }
    struct Raw {
        v4i wh, q0, q1, q2, q3;  // the scales, ql of the two 128s, qh of the two
        uint32_t d;
    };
    __device__ __forceinline__ void read(Raw &R, const uint8_t *slot, int b, int kb, int lane) const {
        R.q0 = *reinterpret_cast<const v4i *>(slot + ql_at + b * 2048);
        R.q1 = *reinterpret_cast<const v4i *>(slot + (ql_at ^ 64u) + b * 2048);
        R.q2 = *reinterpret_cast<const v4i *>(slot + QH + (qh_at ^ (b * 64u)));
        R.q3 = *reinterpret_cast<const v4i *>(slot + QH + (qh_at ^ (b * 64u + 32u)));
        R.wh = *reinterpret_cast<const v4i *>(slot + SC + (sc_at ^ (b * 16u)));
        R.d = *reinterpret_cast<const uint16_t *>(slot + D + (lane & 15) * 16 + ((kb & 7) + b) * 2);
    }
    static __device__ __forceinline__ void arrived(Raw &R) {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(R.wh), "+v"(R.q0), "+v"(R.q1), "+v"(R.q2), "+v"(R.q3), "+v"(R.d)::"memory");
    }
    template <int J>
    static __device__ __forceinline__ void planes(const Raw &R, int g, v4i &H, v4i &L) {
        const v4i nib = J < 2 ? R.q0 : R.q1, two = J < 2 ? R.q2 : R.q3;
        const int s = (int)(int8_t)((uint32_t)R.wh[J] >> (8 * g));
        const uint32_t bias = (uint32_t)(128 - 32 * s), by = 2u * (uint32_t)(g >> 1);
#pragma unroll
        for (int c = 0; c < 4; c++) {
            // the codes' upper two bits: bits 4 (j % 2) + 2 (g / 2) of a byte
            const uint32_t n = (uint32_t)nib[c], t = (uint32_t)two[c] >> by;
            const uint32_t low = (J & 1 ? n >> 4 : n) & 0x0f0f0f0fu, high = (J & 1 ? t : t << 4) & 0x30303030u;
            int h, l;
            byte_planes(low | high, (uint32_t)s, bias, h, l);
            H[c] = h, L[c] = l;
        }
    }
    struct Acts {
        v4i q[4];  // 64j + 16g .. + 15
        v4f d;
    };
    template <bool PLAIN>
    static __device__ __forceinline__ void load_acts(Acts &A, const RowsActs<PLAIN> &a, int kb, int t, int tok, int g) {
        const int at = PLAIN ? tok * a.nb * QK_K + 16 * g : (g >> 1) * 1024 + (g & 1) * 512 + tok * 16;
#pragma unroll
        for (int j = 0; j < 4; j++)
            A.q[j] = __builtin_bit_cast(v4i, __builtin_amdgcn_raw_buffer_load_b128(a.q, at, PLAIN ? kb * QK_K + 64 * j : kb * 8192 + 2048 * j, 0));
        A.d = a.scales(kb, t, g);
    }
    template <int TT>
    static __device__ __forceinline__ void multiply(const Raw &R, int g, const Acts (&A)[TT], v4f (&sum)[TT]) {
        v4i accH[TT], accL[TT];
#pragma unroll
        for (int t = 0; t < TT; t++) accH[t] = accL[t] = v4i{0, 0, 0, 0};
        auto operand = [&](auto j) {
            constexpr int J = decltype(j)::value;
            v4i H, L;
            planes<J>(R, g, H, L);
#pragma unroll
            for (int t = 0; t < TT; t++) {
                accH[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[t].q[J], H, accH[t], 0, 0, 0);
                accL[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[t].q[J], L, accL[t], 0, 0, 0);
            }
        };
        operand(std::integral_constant<int, 0>());
        operand(std::integral_constant<int, 1>());
        operand(std::integral_constant<int, 2>());
        operand(std::integral_constant<int, 3>());
        const float d = h2f(R.d);
#pragma unroll
        for (int t = 0; t < TT; t++)
#pragma unroll
            for (int r = 0; r < 4; r++) sum[t][r] = fmaf(A[t].d[r] * d, (float)((accH[t][r] << 8) + accL[t][r]), sum[t][r]);
    }
};
#else
template <int KIND>
struct RowsSide {  // (the host side needs the slot's size only)
    static constexpr int SLOT = KIND == FRK_KIND_Q4_K ? 16 * 19 * 16 : KIND == FRK_KIND_Q5_K ? 16 * 23 * 16 : 6912;
};
#endif
// Whether the plain rows' quants go through LDS (of Q6_K a lane loads sixteen bytes, in half as many loads), and a wavefront's part of it
template <int KIND, bool PLAIN>
constexpr bool rows_staged() { return PLAIN && KIND != FRK_KIND_Q6_K; }
template <int KIND, bool PLAIN>
constexpr int rows_wave_lds() { return RowsSide<KIND>::SLOT + (rows_staged<KIND, PLAIN>() ? 16 * QK_K : 0); }

// TT tiles of sixteen tokens.  At most 128 registers: two workgroups to a CU (with 180 two tiles took 1.3 to 1.5 times as long).
template <int KIND, int TT, bool PLAIN>
__global__ __launch_bounds__(64 * ROWS_WAVES) __attribute__((amdgpu_waves_per_eu(4))) void gemm_k_rows_kernel(RowsArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
    using Side = RowsSide<KIND>;
    static_assert(Side::SLOT >= TT * 1024 && Side::SLOT == (KIND == FRK_KIND_Q4_K ? 16 * 19 * 16 : KIND == FRK_KIND_Q5_K ? 16 * 23 * 16 : 6912),
                  "a wavefront's sums in its slot; the host's size");
    extern __shared__ __align__(16) uint8_t rows_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6), waves = (int)blockDim.x >> 6;
    const int lr = lane & 15, lq = lane >> 4;
    const int row0 = (int)blockIdx.x * 16;
    constexpr bool STAGED = rows_staged<KIND, PLAIN>();
    static_assert(!STAGED || TT == 1, "sixteen tokens are staged");
    constexpr int WAVE_LDS = rows_wave_lds<KIND, PLAIN>();
    const int pairs = (g.nb + 1) >> 1, p0 = min(wave * g.each, pairs), p1 = min(p0 + g.each, pairs);
    uint8_t *const slot = rows_lds + (size_t)wave * WAVE_LDS;
    const uint32_t slot_lds = lds_address(rows_lds) + (uint32_t)wave * WAVE_LDS;
    const uint8_t *const first = g.W + (size_t)row0 * g.row_stride;
    const Side side(g, lane, min(g.rows - 1 - row0, 15));
    const int tile = (int)blockIdx.y, M = min(g.M - 32 * tile, 32);
    const size_t tile_at = (size_t)tile * 32 * g.nb;
    auto buffer = [&](const void *tiles, const void *rows, int bytes) {  // (bytes a block of a token)
        const uint8_t *const at = PLAIN ? (const uint8_t *)rows : (const uint8_t *)tiles + tile_at * bytes;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(at), 0, (PLAIN ? M : 32) * g.nb * bytes, 0x00027000);
    };
    const RowsActs<PLAIN> acts = {buffer(g.a.q, g.plain.q, 256), buffer(g.a.bs, g.plain.bsums, 32), buffer(g.a.d, g.plain.d, 4), g.nb, M};
    typename Side::Acts A[TT];
    v4f acc[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) acc[t] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    if constexpr (STAGED) {
        const uint8_t *const staged = slot + Side::SLOT;
        const uint32_t staged_lds = slot_lds + Side::SLOT;
        uint32_t from[4];  // (tokens past the batch repeat the last one)
#pragma unroll
        for (int c = 0; c < 4; c++) from[c] = (uint32_t)min(4 * c + lq, M - 1) * (uint32_t)(g.nb * QK_K) + (uint32_t)((lr ^ (4 * c + lq)) * 16);
        typename Side::Small next;
        const int end = min(2 * p1, g.nb);
        auto request = [&](int kb) {
            if (kb < end) Side::stage(staged_lds, g.plain.q, from, kb);
            // (past the share the last block's again: loaded under a condition they would be waited for at its end)
            Side::load_small(next, acts, min(kb, end - 1), min(lr, M - 1), lq);
        };
        if (p0 < p1) {
            side.fetch(g, slot_lds, first, 2 * p0, lane);
            request(2 * p0);
        }
        for (int p = p0; p < p1; p++) {
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const int kb = 2 * p + b;
                if (kb >= g.nb) break;
                // everything asked for so far: this block's quants, sums and scales, at a pair's first block its weights too
                asm volatile("s_waitcnt vmcnt(0)" : "+v"(next.sums), "+v"(next.d)::"memory");
                typename Side::Raw R;
                side.read(R, slot, b, 2 * p, lane);
                Side::take(A[0], next, staged, lane);
                Side::arrived(R);
                // what was read is in registers: the next pair, and the next block's tokens, travel beside the arithmetic
                if (b && p + 1 < p1) side.fetch(g, slot_lds, first, 2 * p + 2, lane);
                request(kb + 1);
                Side::multiply(R, lq, A, acc);
                asm volatile("" : "+v"(acc[0]));  // (in front of the branch, see below)
            }
        }
    } else {
        auto load_acts = [&](int kb) {  // (tokens past the batch repeat the last one)
#pragma unroll
            for (int t = 0; t < TT; t++) Side::load_acts(A[t], acts, kb, t, min(16 * t + lr, M - 1), lq);
        };
        if (p0 < p1) {
            side.fetch(g, slot_lds, first, 2 * p0, lane);
            load_acts(2 * p0);
        }
        for (int p = p0; p < p1; p++) {
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int b = 0; b < 2; b++) {
                const int kb = 2 * p + b;
                if (kb >= g.nb) break;
                typename Side::Raw R;
                side.read(R, slot, b, 2 * p, lane);
                if (b && p + 1 < p1) {
                    // the pair is in registers: the next one travels beside its arithmetic
                    Side::arrived(R);
                    side.fetch(g, slot_lds, first, 2 * p + 2, lane);
                }
                Side::multiply(R, lq, A, acc);
                // (in front of the branch: hipcc counts an MFMA's wait states within a basic block only)
#pragma unroll
                for (int t = 0; t < TT; t++) asm volatile("" : "+v"(acc[t]));
                if (kb + 1 < min(2 * p1, g.nb)) load_acts(kb + 1);
            }
        }
    }
    // register r of lane (row, g): token 4 * g + r
#pragma unroll
    for (int t = 0; t < TT; t++) *reinterpret_cast<v4f *>(slot + t * 1024 + lane * 16) = acc[t];
    __syncthreads();
    for (int i = threadIdx.x; i < 16 * M; i += 64 * waves) {
        const int tok = i >> 4, r = i & 15;
        const uint32_t at = (uint32_t)((tok >> 4) * 1024 + ((tok >> 2 & 3) * 16 + r) * 16 + (tok & 3) * 4);
        float v[ROWS_WAVES];
#pragma unroll
        for (int w = 0; w < ROWS_WAVES; w++) {
            const float one = *reinterpret_cast<const float *>(rows_lds + (size_t)min(w, waves - 1) * WAVE_LDS + at);
            v[w] = w < waves ? one : 0.0f;
        }
        const float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        if (row0 + r < g.rows) g.y[(size_t)(32 * tile + tok) * g.rows + row0 + r] = sum;
    }
#endif
}

// Tiles of 32 rows in the tiled form, straight from the lanes: a wavefront a (row, block), no LDS, no barrier, the last tile's rows past the
// batch left as they are (gemm_k_rows_kernel does not use them).  A workgroup a block, which puts its rows together in LDS and clears
// the tile's others (quantize_q8_k_tiled_kernel), takes 3.6 us at 16 x 4096 where this takes 2.4; the batches of 2 .. 32 rows that
// have it as their first launch, 0.95 of the time.  `plain`: the same quants as plain rows too.
__global__ __launch_bounds__(256) void quantize_q8_k_one_tile_kernel(const float *__restrict__ x, int rows, int nb, Q8KTiled out, Q8KActsOut plain) {
    const int lane = threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    const int at = (int)blockIdx.x * 4 + wave, row = at / nb, kb = at - row * nb;
    if (row >= rows) return;
    const float4 v = reinterpret_cast<const float4 *>(x + ((size_t)row * nb + kb) * QK_K)[lane];
    float d;
    int sum;  // of the 16-wide group
    const uint32_t packed = quantize_q8_k_lane(v, d, sum);
    // slice lane / 8, 16-byte half lane / 4 % 2; the sum of group lane / 4
    const size_t rec = (size_t)(row >> 5) * nb + kb;
    const int at32 = row & 31;
    reinterpret_cast<uint32_t *>(out.q + rec * 8192)[(lane >> 3) * 256 + ((lane >> 2 & 1) * 32 + at32) * 4 + (lane & 3)] = packed;
    if ((lane & 3) == 0) out.bs[rec * 512 + ((lane >> 5) * 32 + at32) * 8 + (lane >> 2 & 7)] = (_Float16)sum;
    if (lane == 0) out.d[rec * 32 + at32] = d;
    if (!plain.q) return;
    reinterpret_cast<uint32_t *>(plain.q + (size_t)at * QK_K)[lane] = packed;
    if ((lane & 3) == 0) plain.bsums[(size_t)at * 16 + (lane >> 2)] = (int16_t)sum;
    if (lane == 0) plain.d[at] = d;
}
int launch_quantize_q8_k_one_tile(const float *x, size_t rows, size_t cols, Q8KTiled out, hipStream_t s, Q8KActsOut plain) {
    const size_t nb = cols / QK_K;
    hipLaunchKernelGGL(quantize_q8_k_one_tile_kernel, dim3((unsigned)((rows * nb + 3) / 4)), dim3(256), 0, s, x, (int)rows, (int)nb, out, plain);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(FRK_ERR_HIP, "quantize_q8_k_one_tile launch: %s", hipGetErrorString(e));
    return FRK_OK;
}

template <int KIND, int TT, bool PLAIN>
static int launch_rows(const RowsArgs &g, dim3 grid, int waves, hipStream_t s) {
    const int lds = waves * rows_wave_lds<KIND, PLAIN>();
    if constexpr (ROWS_WAVES * rows_wave_lds<KIND, PLAIN>() > 65536) {
        static bool sized = false;
        if (!sized) {
            const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_k_rows_kernel<KIND, TT, PLAIN>),
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, ROWS_WAVES * rows_wave_lds<KIND, PLAIN>());
            if (e != hipSuccess) return set_error(FRK_ERR_HIP, "gemm_k_rows setup: %s", hipGetErrorString(e));
            sized = true;
        }
    }
    hipLaunchKernelGGL((gemm_k_rows_kernel<KIND, TT, PLAIN>), grid, dim3(64 * waves), lds, s, g);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(FRK_ERR_HIP, "gemm_k_rows launch: %s", hipGetErrorString(e));
    return FRK_OK;
}
// batch >= 2 from the tiled form (plain null), or up to 32 from plain rows (16 of Q4_K and Q5_K): the same bits.
int launch_gemm_k_rows(const frk_weights *w, int batch, Q8KTiled a, const Q8KActs *plain, float *y, hipStream_t s) {
    RowsArgs g;
    g.W = w->dev;
    g.row_stride = w->layout.row_stride;
    g.off_qh = (uint32_t)w->layout.off_a;
    g.off_sc = (uint32_t)w->layout.off_b;
    g.off_d = (uint32_t)w->layout.off_c;
    g.rows = (int)w->rows;
    g.nb = (int)(w->cols / QK_K);
    g.M = batch;
    g.a = a;
    g.plain = plain ? *plain : Q8KActs{nullptr, nullptr, nullptr};
    g.y = y;
    const int pairs = (g.nb + 1) / 2;
    g.each = (pairs + ROWS_WAVES - 1) / ROWS_WAVES;
    const int waves = (pairs + g.each - 1) / g.each;
    const dim3 grid((unsigned)((w->rows + 15) / 16), (unsigned)((batch + 31) / 32));
#define FRK_GO(KIND, TT, PLAIN) return launch_rows<KIND, TT, PLAIN>(g, grid, waves, s)
#define FRK_GO_KIND(KIND)                         \
    if (plain) FRK_GO(KIND, 1, true);             \
    else if (batch <= 16) FRK_GO(KIND, 1, false); \
    else FRK_GO(KIND, 2, false)
    if (plain && batch > 32) return set_error(FRK_ERR_UNSUPPORTED, "more than 32 plain rows");
    if (w->kind == FRK_KIND_Q6_K) {
        if (plain && batch > 16) FRK_GO(FRK_KIND_Q6_K, 2, true);
        else FRK_GO_KIND(FRK_KIND_Q6_K);
    } else if (plain && batch > 16) {
        return set_error(FRK_ERR_UNSUPPORTED, "more than 16 plain rows of quant kind %d", w->kind);
    } else if (w->kind == FRK_KIND_Q5_K) {
        FRK_GO_KIND(FRK_KIND_Q5_K);
    } else {
        FRK_GO_KIND(FRK_KIND_Q4_K);
    }
#undef FRK_GO_KIND
#undef FRK_GO
}

}  // namespace frk
