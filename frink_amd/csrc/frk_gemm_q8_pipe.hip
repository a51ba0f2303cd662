// The batched Q8_0 GEMM (from 65 rows on; below, gemm_q8_0_rows_kernel): the arithmetic of frk_gemm_q8.hip (an exact int8 MFMA per 32-wide block, the
// block scales' outer product from the f16 matrix core, a conversion and a fused multiply-add per sum, blocks in order),
// over larger tiles that come into LDS without passing through registers.
//
// What bounds it is the issue of the vector ALU beside the matrix core: 32 instructions for a tile's two MFMAs, 64 ns a product
// and SIMD alone (76 in this kernel; the chip holds about 2 GHz under it).  A wavefront owns 32 weight rows and MT tiles
// of 32 tokens, so a weight fragment is read once for MT products (the kernel it replaces read two fragments a product and
// moved 816 bytes a product through registers into LDS; 256 x 128 tiles move 408, and no instruction touches them).
// The columns go by in halves of a chunk (128 columns, four blocks), three stages in LDS, requested two ahead, the
// requests spread over the arithmetic; block scales come a chunk (256 columns) at a time.  One barrier a half chunk, and
// the pipeline of reads, matrix instructions and float steps runs across it: started anew behind every barrier, the wait
// for the first operands and products stood open on both wavefronts of a SIMD (2048 x 4096 x 14336 in tokens x rows x
// columns, with quantization, 310 us; across 301; 512 x 14336 x 4096 87.7 -> 82.7, 200 x 11008 x 4096 46.3 -> 45.5, 512 x
// 4096 x 14336 93.4 -> 90.9).  Tried beside it without gain: the conversion as a subtraction from a sum that starts at 1.5 *
// 2^23 (302), the scales' MFMA in the middle of the float step (303), quants as f16 planes whose sums need no conversion
// (the products alone 60 against 64 ns, for twice the LDS traffic).
#include "frk_device.hpp"

#include <type_traits>

namespace frk {

typedef int qp_v4i __attribute__((ext_vector_type(4)));
typedef int qp_v16i __attribute__((ext_vector_type(16)));
typedef float qp_v16f __attribute__((ext_vector_type(16)));
typedef _Float16 qp_v4h __attribute__((ext_vector_type(4)));

struct Q8PipeArgs {
    const uint8_t *W;  // rows: quants [nb][32], then the f16 scales [nb] at off_d
    size_t row_stride, off_d;
    const int8_t *aq;    // [M][nb * 32]
    const uint16_t *ad;  // [M][nb rounded up to 8], zeros in the padding
    float *y;            // [k_split][M][rows]
    int rows, nb, M;
    int row_tiles, tok_tiles, k_split;
};

// RG x TG wavefronts of 32 rows x MT tiles of tokens
template <int RG, int TG, int MT>
struct Q8PipeLds {
    static_assert(RG * TG == 8, "eight wavefronts");
    static constexpr int ROWS = 32 * RG, TOKS = 32 * TG * MT, LINES = ROWS + TOKS;
    static constexpr int STAGE = LINES * 128, STAGES = 3;
    static constexpr int OFF_SCALES = STAGES * STAGE, SCALES = LINES * 16;  // two slots of a chunk's scales
    static constexpr int REQUESTS = LINES / 64;                            // of a wavefront and half chunk
    static constexpr int SCALE_REQUESTS = LINES / 64;                      // of a chunk, one a wavefront
    static constexpr size_t BYTES = OFF_SCALES + 2 * SCALES;
    static_assert(LINES % 64 == 0 && SCALE_REQUESTS <= 8 && BYTES <= 160 * 1024, "whole requests, LDS of a CU");
};

template <int RG, int TG, int MT>
__global__ __launch_bounds__(512, 2) void gemm_q8_0_pipe_kernel(Q8PipeArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
    using L = Q8PipeLds<RG, TG, MT>;
    constexpr int R = L::REQUESTS;
    extern __shared__ __align__(16) uint8_t qp_lds[];
    const uint32_t lds0 = lds_address(qp_lds);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int li = lane & 31, lg = lane >> 5;
    const int rg = wave % RG, tg = wave / RG;

    // an XCD (block id mod 8) takes a run of the (row tile, token tile) list: its workgroups share weight rows
    const int total = g.row_tiles * g.tok_tiles, per_xcd = (total + 7) / 8;
    const int index = ((int)blockIdx.x & 7) * per_xcd + ((int)blockIdx.x >> 3);
    if (((int)blockIdx.x >> 3) >= per_xcd || index >= total) return;  // (uniform)
    const int row0 = index / g.tok_tiles * L::ROWS, tok0 = index % g.tok_tiles * L::TOKS;
    const int n_chunks = (g.nb + 7) / 8;
    const int chunk0 = n_chunks * (int)blockIdx.y / g.k_split, chunk1 = n_chunks * ((int)blockIdx.y + 1) / g.k_split;
    // half chunks h0 .. h1 - 1 (the last chunk's second half may have no block)
    const int h0 = 2 * chunk0, h1 = min(2 * chunk1, (g.nb + 3) / 4);
    const size_t nbp = (size_t)n_chunks * 8;

    // ---- the requests.  Lines 0 .. ROWS - 1 of a stage are weight rows, the others tokens, 128 bytes each; piece p of
    // line r sits in place p ^ (r / 2) % 8, so that sixteen lines' reads of one piece fall in different banks.  Request n
    // brings lines 8n .. 8n + 7.  (Lines past the operands repeat the last one: their results are not stored.  The last
    // half chunk may reach past a row, into its scales or the next row: those products meet zero scales.  Past the last
    // row there are the resident copy's 256 bytes of slack, and behind the quants of the last token the scales.)
    auto line_offset = [&](int line) -> uint32_t {
        return line < L::ROWS ? (uint32_t)min(row0 + line, g.rows - 1) * (uint32_t)g.row_stride
                              : (uint32_t)min(tok0 + line - L::ROWS, g.M - 1) * (uint32_t)g.nb * 32u;
    };
    uint32_t off[R];
#pragma unroll
    for (int c = 0; c < R; c++) {
        const int line = (wave * R + c) * 8 + (lane >> 3);
        off[c] = line_offset(line) + (uint32_t)((lane & 7) ^ ((line >> 1) & 7)) * 16;
    }
    const bool fetches_scales = wave < L::SCALE_REQUESTS;
    const int scale_line = wave * 64 + lane;  // (64 divides ROWS: a request is all rows or all tokens)
    const uint32_t scale_off = scale_line < L::ROWS ? (uint32_t)min(row0 + scale_line, g.rows - 1) * (uint32_t)g.row_stride
                                                    : (uint32_t)min(tok0 + scale_line - L::ROWS, g.M - 1) * (uint32_t)nbp * 2u;
    const uint8_t *const scale_base = wave * 64 < L::ROWS ? g.W + g.off_d : reinterpret_cast<const uint8_t *>(g.ad);
    int fill = 0;  // the stage the next half chunk goes into
    auto fetch_quants = [&](int h, int c) {
        const int n = wave * R + c;
        const uint8_t *base = 8 * n < L::ROWS ? g.W : reinterpret_cast<const uint8_t *>(g.aq);
        dma16(lds0 + (uint32_t)fill * L::STAGE + (uint32_t)n * 1024, base + (size_t)h * 128, off[c]);
    };
    auto fetch_scales = [&](int h) {  // in front of its chunk's first half
        if (!(h & 1) && fetches_scales)
            dma16(lds0 + L::OFF_SCALES + (uint32_t)((h >> 1) & 1) * L::SCALES + (uint32_t)wave * 1024, scale_base + (size_t)(h >> 1) * 16, scale_off);
    };
    auto filled = [&]() { fill = fill == L::STAGES - 1 ? 0 : fill + 1; };

    qp_v16f acc[MT];
#pragma unroll
    for (int t = 0; t < MT; t++) acc[t] = qp_v16f{0.0f};
    const qp_v16i zero_i = {0};
    const qp_v16f zero_f = {0.0f};
    // this lane's piece of block b in a line of its own row or token, less the line's tile
    uint32_t piece[4];
#pragma unroll
    for (int b = 0; b < 4; b++) piece[b] = (uint32_t)(li * 128 + ((2 * b + lg) ^ ((li >> 1) & 7)) * 16);

#pragma unroll
    for (int ahead = 0; ahead < 2; ahead++)
        if (h0 + ahead < h1) {
            fetch_scales(h0 + ahead);
#pragma unroll
            for (int c = 0; c < R; c++) fetch_quants(h0 + ahead, c);
            filled();
        }
    // ---- A three-stage pipeline over the products (block by block, its MT tiles in turn): the reads of product n + 2, the
    // matrix core's work for n + 1, the float step of n.  It runs across the half chunks: the next one is waited for behind
    // the last product's matrix instructions, its scales and first operands are read in front of the float step before.
    constexpr int N = 4 * MT;
    int at = 0;
    const uint8_t *sw_lines, *sa_lines;
    uint2 sw, sa[MT];  // the four blocks' scales, f16, two to a register; k = 0 of the outer product sits in lanes 0 .. 31
    uint2 sw_next, sa_next[MT];
    auto arrive = [&](int h) {
        // half chunk h (and its chunk's scales) has landed, and everybody has read the one before; behind it only h + 1
        // was requested
        if (h + 1 >= h1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        else if ((h & 1) && fetches_scales) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(R + 1) : "memory");
        else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(R) : "memory");
        lds_barrier();
        const uint8_t *st = qp_lds + (size_t)at * L::STAGE;
        at = at == L::STAGES - 1 ? 0 : at + 1;
        sw_lines = st + rg * 32 * 128;
        sa_lines = st + (L::ROWS + tg * MT * 32) * 128;
        const uint8_t *sc = qp_lds + L::OFF_SCALES + ((h >> 1) & 1) * L::SCALES + (h & 1) * 8;
        sw_next = *reinterpret_cast<const uint2 *>(sc + (rg * 32 + li) * 16);
#pragma unroll
        for (int t = 0; t < MT; t++) sa_next[t] = *reinterpret_cast<const uint2 *>(sc + (L::ROWS + (tg * MT + t) * 32 + li) * 16);
    };
    auto use_scales = [&](int h) {
        const int live = g.nb - 4 * h;  // blocks of the row from here on: a row's scales past its end are whatever lies there
        const uint32_t both = lg ? 0u : 0xffffffffu;
        sw.x = sw_next.x & (live > 1 ? both : both & 0xffffu);
        sw.y = sw_next.y & (live > 3 ? both : live > 2 ? both & 0xffffu : 0u);
#pragma unroll
        for (int t = 0; t < MT; t++) sa[t] = make_uint2(sa_next[t].x & both, sa_next[t].y & both);
    };
    auto k0 = [](uint2 s, int b) {  // {scale of block b, 0, 0, 0}
        const uint32_t w = b < 2 ? s.x : s.y;
        const uint2 u = make_uint2(b & 1 ? w >> 16 : w & 0xffffu, 0u);
        qp_v4h v;
        __builtin_memcpy(&v, &u, 8);
        return v;
    };
    auto read_w = [&](int b) { return *reinterpret_cast<const qp_v4i *>(sw_lines + piece[b]); };
    auto read_a = [&](int n) { return *reinterpret_cast<const qp_v4i *>(sa_lines + (n % MT) * 4096 + piece[n / MT]); };
    qp_v4i w1, w2, a1, a2;
    qp_v16i isum_next;
    qp_v16f scale_next;
    auto multiply = [&](int n) {
        isum_next = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1, w1, zero_i, 0, 0, 0);
        scale_next = __builtin_amdgcn_mfma_f32_32x32x8f16(k0(sa[n % MT], n / MT), k0(sw, n / MT), zero_f, 0, 0, 0);
    };
    // MORE: half chunk h + 2 exists and is requested, NEXT: h + 1 exists.  (Copies of the body instead of branches in it:
    // the compiler counts the wait states between an MFMA and a reader of its result within one basic block only; over the
    // loop's edge 32 vector instructions lie between the two.)
    auto half_chunk = [&](auto more_c, auto next_c, int h) {
        constexpr bool MORE = decltype(more_c)::value, NEXT = decltype(next_c)::value;
        if (MORE) fetch_scales(h + 2);
#pragma unroll
        for (int n = 0; n < N; n++) {
            const qp_v16i isum = isum_next;
            const qp_v16f scale = scale_next;
            if (n == N - 1 && NEXT) use_scales(h + 1);
            if (n + 2 < N) {
                a2 = read_a(n + 2);
                w2 = (n + 2) % MT == 0 ? read_w((n + 2) / MT) : w1;
            }
            if (n + 1 < N || NEXT) multiply((n + 1) % N);
            if (n % (N / R) == 0 && n / (N / R) < R && MORE) fetch_quants(h + 2, n / (N / R));
            if (n == N - 2 && MORE) filled();
            if (n + 2 >= N && NEXT) {
                if (n == N - 2) {
                    __builtin_amdgcn_sched_barrier(0);
                    arrive(h + 1);
                }
                a2 = read_a(n + 2 - N);
                w2 = (n + 2 - N) % MT == 0 ? read_w((n + 2 - N) / MT) : w1;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int r = 0; r < 16; r++) acc[n % MT][r] = __builtin_fmaf(scale[r], (float)isum[r], acc[n % MT][r]);
            asm volatile("" : "+v"(acc[n % MT]));  // (the float step stays here: sunk to the end, every product's sums are alive at once)
            __builtin_amdgcn_sched_barrier(0);
            a1 = a2, w1 = w2;
        }
        static_assert((R - 1) * (N / R) <= N - 2, "a half chunk's requests in front of the next one's wait");
    };
    int h = h0;
    arrive(h0);
    use_scales(h0);
    a1 = read_a(0), w1 = read_w(0);
    a2 = read_a(1), w2 = MT > 1 ? w1 : read_w(1);
    multiply(0);
    a1 = a2, w1 = w2;
    for (; h + 2 < h1; h++) half_chunk(std::true_type(), std::true_type(), h);
    if (h + 1 < h1) half_chunk(std::false_type(), std::true_type(), h++);
    half_chunk(std::false_type(), std::false_type(), h);

    // register r of a lane: token 8 * (r / 4) + 4 * (lane / 32) + r % 4 of the tile, weight row lane % 32
    const int row = row0 + rg * 32 + li;
    float *const dst = g.y + (size_t)blockIdx.y * g.M * g.rows;
    if (row < g.rows) {
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int tok = tok0 + (tg * MT + t) * 32 + 8 * (r >> 2) + 4 * lg + (r & 3);
                if (tok < g.M) dst[(size_t)tok * g.rows + row] = acc[t][r];
            }
    }
#endif
}

// ---- Batches of up to 64 rows: a workgroup is 32 weight rows, its eight wavefronts shares of the columns in order (g.k_split
// workgroups may share a row), whose sums meet in LDS.  The bytes of the weights bound it.  A wavefront brings its rows' and tokens' half
// chunks, whole lines, into a slot of its own with global_load_lds and refills the slot as soon as it is in registers, so nothing
// waits for another wavefront before the end, and rows are rarely split between workgroups, whose sums are a launch more.  TL lines
// of tokens (8, 16, 32, 64 as two tiles; products of lanes past them are not stored): 6 to 13 KB a wavefront, one to three workgroups a CU.
// With quantization (us, tokens x rows x columns; one-wavefront workgroups over registers and LDS copies, in four or eight parts,
// before): 8 x 4096 x 4096 14.2, now 8.0; 8 x 4096 x 14336 22.8, 15.5; 32 x 14336 x 4096 23.2, 15.9; 10 x 1100 x 14336 20.2, 10.5; over 45
// shapes 0.66 of the time in the mean.  With weights past the 256 MB cache 4 x 4096 x 4096 14.7, 9.7, 16 x 14336 x 4096 24.6, 19.2.  33 .. 64
// tokens (four wavefronts over 64 x 64 before): 48 x 14336 x 4096 30.3, 22.3; 30
// shapes 0.73 of the time, 0.84 past the cache.
// Sixteen wavefronts a workgroup, four, two slots a wavefront, non-temporal weights and 64 rows a workgroup were slower or no faster
// over the range; a slot refilled behind the products instead of in front of them 1.2 to 2.7 us slower.
constexpr int ROWS_WAVES = 8;
template <int TL>
struct Q8RowsLds {
    static constexpr int TT = TL > 32 ? 2 : 1;  // tiles of 32 tokens
    static constexpr int TOKENS = 32 * 128, SCALES = TOKENS + TL * 128, TOKEN_SCALES = SCALES + 512, SLOT = TOKEN_SCALES + TT * 512;
    static constexpr size_t BYTES = (size_t)ROWS_WAVES * SLOT;
    static_assert(SLOT >= TT * 4096 && BYTES <= 160 * 1024, "a wavefront's sums in its slots, LDS of a CU");
};
template <int TL>
__global__ __launch_bounds__(64 * ROWS_WAVES) void gemm_q8_0_rows_kernel(Q8PipeArgs g) {
#if defined(__HIP_DEVICE_COMPILE__)
    using L = Q8RowsLds<TL>;
    constexpr int TT = L::TT;
    extern __shared__ __align__(16) uint8_t qp_lds[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int li = lane & 31, lg = lane >> 5;
    const int row0 = (int)blockIdx.x * 32;
    const int halves = (g.nb + 3) / 4, shares = g.k_split * ROWS_WAVES, share = (int)blockIdx.y * ROWS_WAVES + wave;
    const int h0 = (int)((int64_t)halves * share / shares), h1 = (int)((int64_t)halves * (share + 1) / shares);
    const uint32_t nbp = (uint32_t)((g.nb + 7) & ~7);
    uint8_t *const slot = qp_lds + (size_t)wave * L::SLOT;
    const uint32_t slot_lds = lds_address(qp_lds) + (uint32_t)wave * L::SLOT;
    // lines of 128 bytes as in the kernel above: piece p of line r in place p ^ (r / 2) % 8
    uint32_t w_off[4], a_off[TL / 8];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const int line = c * 8 + (lane >> 3);
        w_off[c] = (uint32_t)min(row0 + line, g.rows - 1) * (uint32_t)g.row_stride + (uint32_t)((lane & 7) ^ ((line >> 1) & 7)) * 16;
    }
#pragma unroll
    for (int c = 0; c < TL / 8; c++) {
        const int line = c * 8 + (lane >> 3);
        a_off[c] = (uint32_t)min(line, g.M - 1) * (uint32_t)g.nb * 32u + (uint32_t)((lane & 7) ^ ((line >> 1) & 7)) * 16;
    }
    const uint32_t s_rows = (uint32_t)min(row0 + li, g.rows - 1) * (uint32_t)g.row_stride;
    const uint32_t s_tokens = (uint32_t)min(TT == 2 ? lane : li, g.M - 1) * nbp * 2u;
    const uint8_t *const ad = reinterpret_cast<const uint8_t *>(g.ad);
    auto request = [&](int h) {
#pragma unroll
        for (int c = 0; c < 4; c++) dma16(slot_lds + c * 1024, g.W + (size_t)h * 128, w_off[c]);
#pragma unroll
        for (int c = 0; c < TL / 8; c++) dma16(slot_lds + L::TOKENS + c * 1024, reinterpret_cast<const uint8_t *>(g.aq) + (size_t)h * 128, a_off[c]);
        const size_t at = (size_t)(h >> 1) * 16;  // (a chunk's scales, with each of its halves)
        if (!lg) dma16(slot_lds + L::SCALES, g.W + g.off_d + at, s_rows);
        if (TT == 2) dma16(slot_lds + L::TOKEN_SCALES, ad + at, s_tokens);
        else if (lg) dma16(slot_lds + L::SCALES, ad + at, s_tokens);  // (lane 32 is 512 bytes further)
    };
    qp_v16f acc[TT];
#pragma unroll
    for (int t = 0; t < TT; t++) acc[t] = qp_v16f{0.0f};
    const qp_v16i zero_i = {0};
    const qp_v16f zero_f = {0.0f};
    if (h0 < h1) request(h0);
    for (int h = h0; h < h1; h++) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        uint2 sw = *reinterpret_cast<const uint2 *>(slot + L::SCALES + li * 16 + (h & 1) * 8);
        uint2 sa[TT];
        qp_v4i w[4], a[TT][4];
#pragma unroll
        for (int t = 0; t < TT; t++) sa[t] = *reinterpret_cast<const uint2 *>(slot + L::TOKEN_SCALES + (32 * t + li) * 16 + (h & 1) * 8);
#pragma unroll
        for (int b = 0; b < 4; b++) {
            w[b] = *reinterpret_cast<const qp_v4i *>(slot + li * 128 + ((2 * b + lg) ^ ((li >> 1) & 7)) * 16);
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const int line = 32 * t + (li & (TL - 1));
                a[t][b] = *reinterpret_cast<const qp_v4i *>(slot + L::TOKENS + line * 128 + ((2 * b + lg) ^ ((line >> 1) & 7)) * 16);
            }
        }
        // the slot is in registers: the next half chunk travels beside the arithmetic
#pragma unroll
        for (int t = 0; t < TT; t++) asm volatile("" : "+v"(sa[t]), "+v"(a[t][0]), "+v"(a[t][1]), "+v"(a[t][2]), "+v"(a[t][3]));
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(sw), "+v"(w[0]), "+v"(w[1]), "+v"(w[2]), "+v"(w[3])::"memory");
        if (h + 1 < h1) request(h + 1);
        const int live = g.nb - 4 * h;  // blocks of the row from here on: behind its end lie other bytes
        const uint32_t both = lg ? 0u : 0xffffffffu;
        sw.x &= live > 1 ? both : both & 0xffffu;
        sw.y &= live > 3 ? both : live > 2 ? both & 0xffffu : 0u;
#pragma unroll
        for (int t = 0; t < TT; t++) sa[t].x &= both, sa[t].y &= both;
        auto k0 = [](uint2 s, int b) {
            const uint32_t v = b < 2 ? s.x : s.y;
            const uint2 u = make_uint2(b & 1 ? v >> 16 : v & 0xffffu, 0u);
            qp_v4h o;
            __builtin_memcpy(&o, &u, 8);
            return o;
        };
#pragma unroll
        for (int b = 0; b < 4; b++)
#pragma unroll
            for (int t = 0; t < TT; t++) {
                const qp_v16i isum = __builtin_amdgcn_mfma_i32_32x32x32_i8(a[t][b], w[b], zero_i, 0, 0, 0);
                const qp_v16f scale = __builtin_amdgcn_mfma_f32_32x32x8f16(k0(sa[t], b), k0(sw, b), zero_f, 0, 0, 0);
#pragma unroll
                for (int r = 0; r < 16; r++) acc[t][r] = __builtin_fmaf(scale[r], (float)isum[r], acc[t][r]);
            }
    }
    // register r of a lane: token 8 * (r / 4) + 4 * (lane / 32) + r % 4, weight row lane % 32
#pragma unroll
    for (int t = 0; t < TT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) reinterpret_cast<float *>(slot)[t * 1024 + r * 64 + lane] = acc[t][r];
    __syncthreads();
    float *const dst = g.y + (size_t)blockIdx.y * g.M * g.rows;
    for (int i = threadIdx.x; i < 32 * g.M; i += 64 * ROWS_WAVES) {
        const int tok = i >> 5, row = i & 31;
        const int at = (tok >> 5) * 1024 + ((tok >> 3 & 3) * 4 + (tok & 3)) * 64 + ((tok >> 2) & 1) * 32 + row;
        float sum = 0.0f;
#pragma unroll
        for (int v = 0; v < ROWS_WAVES; v++) {
            const float one = reinterpret_cast<const float *>(qp_lds + (size_t)v * L::SLOT)[at];
            sum = v ? sum + one : one;
        }
        if (row0 + row < g.rows) dst[(size_t)tok * g.rows + row0 + row] = sum;
    }
#endif
}
template <int TL>
static int launch_rows(const Q8PipeArgs &g, hipStream_t s) {
    using L = Q8RowsLds<TL>;
    static bool sized = false;  // a benign race: every thread sets the same attribute
    if (!sized) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_q8_0_rows_kernel<TL>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::BYTES);
        if (e != hipSuccess) return set_error(FRK_ERR_HIP, "hipFuncSetAttribute(LDS %zu): %s", L::BYTES, hipGetErrorString(e));
        sized = true;
    }
    hipLaunchKernelGGL((gemm_q8_0_rows_kernel<TL>), dim3((unsigned)((g.rows + 31) / 32), (unsigned)g.k_split), dim3(64 * ROWS_WAVES), L::BYTES, s, g);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(FRK_ERR_HIP, "gemm_q8_0_rows launch: %s", hipGetErrorString(e));
    return FRK_OK;
}

template <int RG, int TG, int MT>
static int launch_tile(const Q8PipeArgs &g, hipStream_t s) {
    using L = Q8PipeLds<RG, TG, MT>;
    static bool sized = false;  // a benign race: every thread sets the same attribute
    if (!sized) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&gemm_q8_0_pipe_kernel<RG, TG, MT>),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::BYTES);
        if (e != hipSuccess) return set_error(FRK_ERR_HIP, "hipFuncSetAttribute(LDS %zu): %s", L::BYTES, hipGetErrorString(e));
        sized = true;
    }
    const unsigned grid = (unsigned)((g.row_tiles * g.tok_tiles + 7) / 8 * 8);
    hipLaunchKernelGGL((gemm_q8_0_pipe_kernel<RG, TG, MT>), dim3(grid, (unsigned)g.k_split), dim3(512), L::BYTES, s, g);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(FRK_ERR_HIP, "gemm_q8_0_pipe launch: %s", hipGetErrorString(e));
    return FRK_OK;
}

// The split of gemm_q8_0_rows_kernel: rounds of workgroups over 256 CUs times a wavefront's half chunks (0.9 us each with 8 lines of
// tokens, 1.1 with 16, 1.35 with 32, 2.2 with 64) against the second launch and the parts' bytes.  Measured (us; 1, 2, 4 workgroups a row, tokens x
// rows x columns): 8 x 4096 x 4096 8.0, 10.3, 10.6; 8 x 4096 x 14336 17.2, 15.5, 15.5; 16 x 1500 x 8192 12.6, 10.5, 10.3; 16 x 10240 x
// 10240 41.2, 34.5, 34.3; 32 x 14336 x 4096 15.9, 18.5, 20.5.
static Q8PipePlan q8_rows_plan(size_t rows, size_t M, size_t nb, size_t max_parts) {
    const size_t groups = (rows + 31) / 32, halves = (nb + 3) / 4;
    const int lines = M <= 8 ? 8 : M <= 16 ? 16 : M <= 32 ? 32 : 64;
    const double step = lines == 8 ? 0.9 : lines == 16 ? 1.1 : lines == 32 ? 1.35 : 2.2;
    Q8PipePlan best = {32, lines, 1};
    double least = 0.0;
    for (size_t ks = 1; ks <= 8 && (ks == 1 || (ks <= max_parts && halves >= 8 * ks)); ks *= 2) {
        double us = (double)((groups * ks + 255) / 256) * (double)((halves + 8 * ks - 1) / (8 * ks)) * step;
        if (ks > 1) us += 3.0 + (double)(2 * ks + 1) * (double)(M * rows) * 4.0 / 6.2e6;
        if (ks == 1 || us < least) least = us, best.k_split = (int)ks;
    }
    return best;
}

// The tile and the split by estimated time, in us, `old_us` (without what all forms share) being the other kernel's.
// Measured a half chunk (one workgroup a CU, one round of the chip): 256 x 128 tiles 2.64, 128 x 64 tiles 0.85 alone and
// 1.47 in pairs (two fit a CU), the other kernel's 64 x 128 tiles 0.84 -- a 128 x 64 share of the work costs 0.66, 0.73 and
// 0.84; a split's parts move at 6.2 TB/s.  With quantization, other kernel -> this one: 2048 x 4096 x 14336 388 -> 317 us,
// 512 x 14336 x 4096 113 -> 91, 200 x 11008 x 4096 62 -> 49, 512 x 4096 x 14336 107 -> 98, 1000 x 4096 x 4096 64 -> 58;
// grids of one round of the other kernel (2048 x 1024 x 4096: 40 against 42 us) stay there.
Q8PipePlan q8_pipe_plan(size_t rows, size_t M, size_t nb, size_t row_stride, int old_split, size_t max_parts) {
    Q8PipePlan best = {0, 0, 0};
    // (Past 80 M weights the other kernel stays for 9 .. 32 and 45 .. 64 tokens, whose tiles it fills: there every workgroup's reads of all tokens cost what the sum's launch
    // did; 32 x 6000 x 13824 34.9 us, here 40.2, 16 x 14314 x 9984 47.9 and 50.2, but 4 x 6000 x 13824 32.8 and 30.4, 32 x 8000 x 8960
    // 32.2 and 29.9; 33, 48 and 64 x 14314 x 9984 66.5 and 61.7, 66.9 and 68.0, 67.3 and 73.7; all from memory.)
    if (M <= 64 && (M <= 8 || (M > 32 && M <= 44) || rows * nb * 32 <= (size_t)80 << 20) && rows * row_stride <= 0xffffffffu && M * nb * 32 <= 0xffffffffu)
        return q8_rows_plan(rows, M, nb, max_parts);
    if (M <= 64 || rows * row_stride > 0xffffffffu || M * nb * 32 > 0xffffffffu) return best;  // (32-bit lane offsets)
    auto tiles = [](size_t n, size_t t) { return (n + t - 1) / t; };
    auto parts = [&](size_t ks) { return ks > 1 ? 3.0 + (double)(2 * ks + 1) * (double)(M * rows) * 4.0 / 6.2e6 : 0.0; };
    const size_t halves = (nb + 3) / 4, chunks = (nb + 7) / 8;
    const double old_us = (double)tiles(tiles(rows, 64) * tiles(M, 128) * (size_t)old_split, 256) * 0.84 * (double)halves / old_split + parts(old_split);
    double least = 0.97 * old_us - 2.0;  // (and two more to start)
    for (size_t ks = 1; ks <= 4 && chunks / ks >= 2; ks *= 2) {
        if (ks > 1 && ks > max_parts) break;
        const double steps = (double)(2 * tiles(chunks, ks));
        const size_t large = tiles(rows, 256) * tiles(M, 128) * ks, small = tiles(rows, 128) * tiles(M, 64) * ks, rest = small % 512;
        const double large_us = (double)tiles(large, 256) * 2.64 * steps + parts(ks);
        const double small_us = ((double)(small / 512) * 1.47 + (rest == 0 ? 0.0 : rest <= 256 ? 0.85 : 1.47)) * steps + parts(ks);
        if (large_us < least) least = large_us, best = Q8PipePlan{256, 128, (int)ks};
        if (small_us < least) least = small_us, best = Q8PipePlan{128, 64, (int)ks};
    }
    return best;
}
int launch_gemm_q8_0_pipe(const Q8PipePlan &p, const uint8_t *W, size_t row_stride, size_t off_d, size_t rows, size_t nb,
                          const int8_t *aq, const uint16_t *ad, size_t M, float *y, hipStream_t s) {
    Q8PipeArgs g;
    g.W = W;
    g.row_stride = row_stride;
    g.off_d = off_d;
    g.aq = aq;
    g.ad = ad;
    g.y = y;
    g.rows = (int)rows;
    g.nb = (int)nb;
    g.M = (int)M;
    g.row_tiles = (int)((rows + p.rows_wg - 1) / p.rows_wg);
    g.tok_tiles = (int)((M + p.tok_wg - 1) / p.tok_wg);
    g.k_split = p.k_split;
    if (p.rows_wg == 32) return p.tok_wg == 8 ? launch_rows<8>(g, s) : p.tok_wg == 16 ? launch_rows<16>(g, s) : p.tok_wg == 32 ? launch_rows<32>(g, s) : launch_rows<64>(g, s);
    if (p.rows_wg == 256) return launch_tile<8, 1, 4>(g, s);
    return launch_tile<4, 2, 1>(g, s);
}

}  // namespace frk
