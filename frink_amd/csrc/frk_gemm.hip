// Prefill / batched GEMM over Q4_K weights on the matrix cores:
//   y[tok][row] = sum_k W[row][k] * x[tok][k],  x quantized per token to Q8_K first.
//
// Arithmetic is dot_q4_k_q8's (crates/frink-quant/src/lib.rs:822-869), regrouped so that a whole
// 256-weight block accumulates inside the MFMA:
//   S1 = sum_j sc_j * isum_j   with sc_j = 8*sh_j + sl_j (sh, sl < 8): a weight row's block becomes two
//                              int8 operand planes  H = sh_j * q  and  L = sl_j * q  (each < 106), so
//                              S1 = 8 * (acts . H) + (acts . L), exact, no per-sub-block rescale;
//   S2 = sum_j m_j * bsum_j    the activation's 16-wide sums (|bsum| <= 2032) and the 6-bit mins are both
//                              exact in f16, their products and the 16-term sum exact in f32, so one
//                              v_mfma_f32_32x32x16_f16 gives S2 already as a float.
// Per block and output the epilogue is then  acc += da * (d * S1 - dmin * S2)  in f32.
// (Scaling each sub-block's product after a K=32 MFMA instead -- one v_mad_i32_i24 per result and
// sub-block -- was measured slower here: it is bound by the vector ALU and needs more registers.)
//
// MFMA operand roles: A = activations (tile row = token), B = weights (tile column = weight row), so
// a lane's 16 results share one weight row (its d, dmin are per-lane values) and span 16 tokens.
// Operand layout of v_mfma_i32_32x32x32_i8 (checked on the device): lane l holds, for row/column
// l % 32, the 16 k-values 16*(l/32) .. +15 (8*(l/32) .. +7 for the K=16 f16 form); result register
// r of lane l is D[8*(r/4) + 4*(l/32) + r%4][l % 32].
//
// Data movement: everything a block needs -- the workgroup's weight rows (raw blocks) and its
// activation tile -- goes from global memory straight into LDS with global_load_lds_dwordx4
// (the 64 lanes' 16-byte pieces land in 1 KB of consecutive LDS; each lane chooses which piece it
// fetches, so the LDS image is whatever order the consumer wants), several blocks ahead, in rings of
// stages.  No prefetch lives in registers, and the only waits on memory are "the stage issued P
// iterations ago has landed".
#include "frk_gemm_pipe.hpp"

namespace frk {

// Activation side: Q8_K quantization (quantize_activations_q8_k, crates/frink-quant/src/act_quant.rs:69-104)
// into the tiled form, one workgroup per record (32 rows x one block).
// Without `gather`, out row r = x[r] (rows from `rows` to the end of the last tile become zeros); with
// it, out row r = x[gather[r]] (zeros where the entry is negative) for the records whose first entry
// is not negative.
// `plain` (without `gather`): the same quants as plain rows too, for a batch whose matrices read either form -- one launch
// where there were two (17 .. 64 rows of 4096 .. 14336 columns 10.3 -> 7.3 us; launch-bound).
template <int WAVES>
__global__ __launch_bounds__(64 * WAVES) void quantize_q8_k_tiled_kernel(const float *__restrict__ x, int rows, int nb,
                                                                  const int *__restrict__ gather, Q8KTiled out, Q8KActsOut plain) {
    __shared__ Q8KRecordLds L;
    const int t32 = blockIdx.x / nb, kb = blockIdx.x % nb, lane = threadIdx.x & 63;
    if (gather && gather[t32 * 32] < 0) return;
    quantize_q8k_record<WAVES>(out, (size_t)t32 * nb + kb, L, [&](int r) {
        const int row = t32 * 32 + r;
        const int src = gather ? gather[row] : (row < rows ? row : -1);
        if (src < 0) return make_float4(0.f, 0.f, 0.f, 0.f);
        return reinterpret_cast<const float4 *>(x + ((size_t)src * nb + kb) * QK_K)[lane];
    }, [&](int r, uint32_t packed, float d, int sum) {
        const int row = t32 * 32 + r;
        if (!plain.q || row >= rows) return;
        const size_t b = (size_t)row * nb + kb;
        reinterpret_cast<uint32_t *>(plain.q + b * QK_K)[lane] = packed;
        if ((lane & 3) == 0) plain.bsums[b * 16 + (lane >> 2)] = (int16_t)sum;
        if (lane == 0) plain.d[b] = d;
    });
}

// The same without `gather`, straight from the lanes: a wavefront a (row, block), no LDS, no barrier.  A workgroup is eight rows of a block, whose
// sixteen-byte pieces and sums are whole lines of 128 bytes (with four blocks of one row a workgroup, lines are put together from
// eight CUs' stores: 512 x 14336 11.7 us where this takes 8.9).
__global__ __launch_bounds__(512) void quantize_q8_k_octets_kernel(const float *__restrict__ x, int rows, int nb, Q8KTiled out, Q8KActsOut plain) {
    const int lane = threadIdx.x & 63, wave = (int)threadIdx.x >> 6;
    const int octet = (int)blockIdx.x / nb, kb = (int)blockIdx.x - octet * nb, row = octet * 8 + wave;
    const size_t at = (size_t)row * nb + kb;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (row < rows) v = reinterpret_cast<const float4 *>(x + at * QK_K)[lane];
    float d;
    int sum;  // of the 16-wide group
    const uint32_t packed = quantize_q8_k_lane(v, d, sum);
    // slice lane / 8, 16-byte half lane / 4 % 2; the sum of group lane / 4
    const size_t rec = (size_t)(row >> 5) * nb + kb;
    const int at32 = row & 31;
    reinterpret_cast<uint32_t *>(out.q + rec * 8192)[(lane >> 3) * 256 + ((lane >> 2 & 1) * 32 + at32) * 4 + (lane & 3)] = packed;
    if ((lane & 3) == 0) out.bs[rec * 512 + ((lane >> 5) * 32 + at32) * 8 + (lane >> 2 & 7)] = (_Float16)sum;
    if (lane == 0) out.d[rec * 32 + at32] = d;
    if (!plain.q || row >= rows) return;
    reinterpret_cast<uint32_t *>(plain.q + at * QK_K)[lane] = packed;
    if ((lane & 3) == 0) plain.bsums[at * 16 + (lane >> 2)] = (int16_t)sum;
    if (lane == 0) plain.d[at] = d;
}

// The grouped form: work items (tile, matrix, row group of 128 rows) streamed by persistent workgroups.
struct StreamArgs {
    const uint8_t *W[2];
    float *y[2];  // row (tile's first row of y + r) x [rows]: tile row r
    int n_mat;
    size_t row_stride;
    uint32_t off_qh, off_sc, off_d;  // the planes of a Q6_K row
    int rows, nb;                    // of one expert
    Q8KTiled a;
    const int4 *tiles;  // {expert, first row of the grouped order, rows in use, first row of y}
    const int *n_tiles;
    int row_tiles;  // ceil(rows / 128)
    // the gathering form: the activations are the source rows' Q8_K, quantized once each, and row r of the
    // grouped order is source row gather[r] (negative: a row not in use)
    Q8KRows src;
    const int *gather;
};

struct TileAcc {
    v16i s1;  // sum_j sc_j * isum_j
    v16f s2;  // sum_j m_j * bsum_j
};

template <bool SUMS>
__device__ __forceinline__ void read_ops(TileOperands &T, uint32_t quants, uint32_t bsums) {
    FRK_DS_READ(T.a0, quants, 0);
    FRK_DS_READ(T.a1, quants, 1024);
    FRK_DS_READ(T.a2, quants, 2048);
    FRK_DS_READ(T.a3, quants, 3072);
    FRK_DS_READ(T.a4, quants, 4096);
    FRK_DS_READ(T.a5, quants, 5120);
    FRK_DS_READ(T.a6, quants, 6144);
    FRK_DS_READ(T.a7, quants, 7168);
    if (SUMS) FRK_DS_READ(T.bs, bsums, 0);
}
template <bool MINS>
__device__ __forceinline__ void tile_epilogue(const TileAcc &X, const TileScales &S, const BPlanes &B, v16f &acc) {
    const v4f dav[4] = {S.da0, S.da1, S.da2, S.da3};
#pragma unroll
    for (int c = 0; c < 4; c++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
            const int r = c * 4 + e;
            if (MINS) {
                const float v = fmaf(B.ndmin, X.s2[r], B.d * (float)X.s1[r]);
                acc[r] = fmaf(dav[c][e], v, acc[r]);
            } else {
                acc[r] = fmaf(dav[c][e] * B.d, (float)X.s1[r], acc[r]);
            }
        }
}

// The 16 + 1 MFMAs of a tile, each waiting only for the operand it needs: the tile's nine LDS reads
// (a0..a7, bs, in that order) must be the wavefront's youngest LDS operations.
// (Each wait also names the running sum as modified, which pins it between its two MFMAs: without
// that the MFMAs are free to sink below all the waits, and the chain starts only when the last
// operand is there.)
template <int N, class V>
__device__ __forceinline__ void wait_lgkm(V &reg, v16i &acc) {
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(reg), "+v"(acc) : "n"(N));
}
// between(i, acc) is called after MFMA i of the integer chain has been issued, i = 0..14: what it does
// shares the gaps of the chain, every MFMA of which waits for the one before it.  It must not branch:
// hipcc counts the wait states between an MFMA and a vector instruction that reads its result within
// one basic block only, and a branch between MFMA 7 and the shift of its sums left the shift three
// instructions behind the MFMA (the last two registers of the sums were read before they were written).
struct NothingBetween {
    __device__ __forceinline__ void operator()(int, v16i &) const {}
};
template <bool MINS, int SHIFT, class Between = NothingBetween>
__device__ __forceinline__ void tile_mfmas_as_they_land(TileOperands &T, const BPlanes &B, TileAcc &X,
                                                        Between between = Between()) {
    const v16i zi = {0};
    const v16f zf = {0.0f};
    constexpr int LATER = MINS ? 1 : 0;
    asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(T.a0) : "n"(7 + LATER));
    v16i acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a0, B.H0, zi, 0, 0, 0);
    between(0, acc);
    wait_lgkm<6 + LATER>(T.a1, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a1, B.H1, acc, 0, 0, 0);
    between(1, acc);
    wait_lgkm<5 + LATER>(T.a2, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a2, B.H2, acc, 0, 0, 0);
    between(2, acc);
    wait_lgkm<4 + LATER>(T.a3, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a3, B.H3, acc, 0, 0, 0);
    between(3, acc);
    wait_lgkm<3 + LATER>(T.a4, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a4, B.H4, acc, 0, 0, 0);
    between(4, acc);
    wait_lgkm<2 + LATER>(T.a5, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a5, B.H5, acc, 0, 0, 0);
    between(5, acc);
    wait_lgkm<1 + LATER>(T.a6, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a6, B.H6, acc, 0, 0, 0);
    between(6, acc);
    wait_lgkm<LATER>(T.a7, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a7, B.H7, acc, 0, 0, 0);
    between(7, acc);
    if constexpr (MINS) {
        wait_lgkm<0>(T.bs, acc);
        X.s2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(T.bs, B.m, zf, 0, 0, 0);
    }
    acc = acc << SHIFT;
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a0, B.L0, acc, 0, 0, 0);
    between(8, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a1, B.L1, acc, 0, 0, 0);
    between(9, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a2, B.L2, acc, 0, 0, 0);
    between(10, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a3, B.L3, acc, 0, 0, 0);
    between(11, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a4, B.L4, acc, 0, 0, 0);
    between(12, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a5, B.L5, acc, 0, 0, 0);
    between(13, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a6, B.L6, acc, 0, 0, 0);
    between(14, acc);
    X.s1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a7, B.L7, acc, 0, 0, 0);
}

template <int RG, int KS, int MT>
__global__ __launch_bounds__(512) void gemm_q4_k_pipe_kernel(GemmArgs g) {
    pipe_gemm<FRK_KIND_Q4_K, RG, KS, MT>(g);
}
template <int RG, int KS, int MT>
__global__ __launch_bounds__(512) void gemm_q5_k_pipe_kernel(GemmArgs g) {
    pipe_gemm<FRK_KIND_Q5_K, RG, KS, MT>(g);
}

// The grouped (per-expert) GEMM: with a few dozen activation rows per expert the work is a stream
// over the experts' weights.  Persistent workgroups (two per CU, 4 wavefronts, 128 weight rows) walk
// a list of work items (tile, matrix, row group); one step = one 256-wide block of one item.  A
// step's data travels into LDS ahead of it, across item boundaries: the weights two or three steps (a wavefront
// fetches and reads only its own 32 rows, so that ring needs no barrier: two stages, Q6_K one, each refilled as
// soon as its block has left it for the registers) and the tile's activation record one step (shared, two
// stages, one barrier per step).  A tile is up to 64 activation rows, two 32-row halves that share
// the unpacked weights; the second half is neither fetched nor multiplied when not in use.
// (One workgroup of 8 wavefronts and 256 rows a CU, activations three steps ahead, had every wavefront of the CU wait for
// the slowest at every step, and items half as many: where they did not fill the chip, 23.1 -> 17.6 us for gate and up of 16
// experts of 1792 / 512 over 540 pairs, 29.7 -> 24.2 over 1494 of 2304 / 512; Q6_K down experts of 128 x 2048 x 768 over
// 4096 pairs 63.9 -> 59, the layer's gate and up as before.  36 drawn layers of 32 to 1024 tokens 0.92 of the time in the
// mean, 0.84 at best, 1.014 at most.)
// The unpacked weights are double-buffered in registers: step s+1 is unpacked from inside the chain
// of MFMAs of step s.  Half of a workgroup's wavefronts ask for their weights before the MFMAs and half
// after: a wavefront is stalled while its loads wait for the CU's address unit, and this way others have the
// matrix cores meanwhile (all before: 1 % on the layer's time; all after: 0.5).
// Items of a tile sit on one XCD (block id mod 8), whose L2 then serves the tile's activations.
// GATHER: a tile's activation rows are fetched from where their source rows were quantized (plain rows,
// each quantized once however many tiles it is part of) instead of from a record of the grouped order: a
// lane's piece of a record is 16 bytes of one row in either form, so only the lane offsets differ -- the
// source row times the row length, looked up per item from a table in LDS.
// KIND: Q4_K or Q6_K.  A Q6_K block is half as large again: one stage of weights, two steps ahead.  (Q6_K down experts of
// 128 x 2048 x 768, 4096 pairs, 165 MB of weights: the dense kernel by tile, one workgroup per tile and 256 rows with
// its three blocks, took 99 us.)
template <int KIND, bool GATHER>
struct StreamLds {
    using Side = WeightSide<KIND>;
    static constexpr bool MINS = Side::MINS;
    static constexpr int RG = 4;
    static constexpr int W_WAVE = Side::SLOT;    // a wavefront's 32 rows of one block
    static constexpr int W_STAGE = RG * W_WAVE;
    static constexpr int W_STAGES = KIND == FRK_KIND_Q6_K ? 1 : 2;
    static constexpr int A_BS = 8192, A_DA = MINS ? 9216 : 8192;  // record of 32 rows: quants | sums (with mins) | scales
    static constexpr int A_HALF = A_DA + 256;  // (64 lanes fetch the 32 scales twice)
    static constexpr int A_STAGE = 2 * A_HALF;   // a tile is two records
    static constexpr int A_STAGES = 2;
    static constexpr int OFF_A = W_STAGES * W_STAGE;
    // {expert, rows in use | matrix << 7 | row group << 8, first row of y, tile} of each of the workgroup's items, filled
    // once: looked up from LDS, an item change costs no global load (whose completion would count in vmcnt, in the
    // middle of the prefetch bookkeeping) and no division (a wavefront's end of step waits for it)
    static constexpr int OFF_ITEMS = OFF_A + A_STAGES * A_STAGE;
    static constexpr int MAX_ITEMS = GATHER ? 28 : 128;
    // GATHER: the source rows of each item's tile, row r of the first half in the low 16 bits of word r and
    // row 32 + r in the high ones
    static constexpr int OFF_SRC = OFF_ITEMS + MAX_ITEMS * 16;
    static constexpr size_t BYTES = (size_t)OFF_SRC + (GATHER ? MAX_ITEMS * 128 : 0);
    static_assert(BYTES <= 80 * 1024, "two workgroups share the LDS of a CU");
};

template <int KIND, bool GATHER>
__device__ __forceinline__ void stream_gemm(const StreamArgs &g) {
    using L = StreamLds<KIND, GATHER>;
    using Side = typename L::Side;
    constexpr bool MINS = L::MINS;
    extern __shared__ uint4 smem_gemm[];
    uint8_t *lds = reinterpret_cast<uint8_t *>(smem_gemm);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lg = lane >> 5;
    const int nb = g.nb;

    // this workgroup's items: the list of its XCD holds the tiles t = xcd (mod 8), every (matrix, row
    // group) of a tile in a row; the XCD's workgroups take list entries slot, slot + per_xcd, ...
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3, per_xcd = gridDim.x >> 3;
    const int n_tiles = *g.n_tiles;
    const int per_tile = g.n_mat * g.row_tiles;
    const int list_len = (n_tiles > xcd ? (n_tiles - xcd + 7) / 8 : 0) * per_tile;
    const int my_items = list_len > slot ? (list_len - slot + per_xcd - 1) / per_xcd : 0;
    const int total_steps = my_items * nb;
    if (total_steps == 0) return;
    {
        int4 *table = reinterpret_cast<int4 *>(lds + L::OFF_ITEMS);
        for (int i = tid; i < my_items; i += 64 * L::RG) {
            const int j = slot + i * per_xcd, t = xcd + 8 * (j / per_tile), w = j % per_tile;
            const int4 ti = g.tiles[t];
            table[i] = make_int4(ti.x, ti.z | (w / g.row_tiles) << 7 | (w % g.row_tiles) << 8, ti.w, t);
        }
        if (GATHER) {
            uint32_t *src_rows = reinterpret_cast<uint32_t *>(lds + L::OFF_SRC);
            for (int i = tid; i < my_items * 32; i += 64 * L::RG) {
                const int t = xcd + 8 * ((slot + (i >> 5) * per_xcd) / per_tile), r = i & 31;
                const int a = g.gather[t * MOE_TILE + r], b = g.gather[t * MOE_TILE + 32 + r];
                src_rows[i] = (uint32_t)max(a, 0) | ((uint32_t)max(b, 0) << 16);  // (a row not in use: any row will do)
            }
        }
        __syncthreads();
    }
    const uint32_t lds_items = lds_address(lds + L::OFF_ITEMS);
    struct Item {
        int tile, expert, mat, row_group, count, y_row;  // (uniform)
    };
    auto item = [&](int ord) {
        v4i v;
        asm volatile("ds_read_b128 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(v) : "v"(lds_items + ord * 16));
        const int y = __builtin_amdgcn_readfirstlane(v.y);
        return Item{__builtin_amdgcn_readfirstlane(v.w), __builtin_amdgcn_readfirstlane(v.x), (y >> 7) & 1, y >> 8, y & 127,
                    __builtin_amdgcn_readfirstlane(v.z)};
    };

    // ---- the fetch side: two cursors (item, block).  While step s is multiplied the activations' asks for step s + 1
    // (A_STAGES is 2: the stage that step s - 1 was read from, which the barrier at its end has freed) and the weights' for
    // step s + 1 + W_STAGES, into the stage that step s + 1's block has just left for the registers: three steps ahead, Q6_K two.
    // weights of a step: this wavefront's 32 rows (WeightSide), which no other wavefront reads.  Addresses are a uniform base
    // that moves with the cursor plus a lane offset: the activations' is fixed per item, the weights' for the kernel (recomputing
    // the offsets from the lane number cost ~60 vector instructions per step, and per item still 2 % of a layer).
    Side wside;
    auto opaque_lane = [&]() {  // the lane number as a value the compiler cannot hoist expressions of
        int l = lane;
        asm volatile("" : "+v"(l));
        return l;
    };
    // activations: quant slices `wave` and `wave` + 4 of each half in use, plus one of the four small pieces: sums
    // (wavefronts 0, 2; only with mins) and scales (1, 3) of the first (0, 1) and second half (2, 3)
    const bool x_sums = (wave & 1) == 0;
    const bool x_small = wave < 4 && (MINS || !x_sums), x_second = wave >= 2;  // fetches a small piece at all; the second half's
    uint32_t qa_off, qb_off, x_off;
    if (!GATHER) {
        qa_off = (uint32_t)(wave * 1024 + lane * 16);
        qb_off = qa_off + (uint32_t)nb * 8192;
        x_off = x_sums ? (uint32_t)lane * 16 : (uint32_t)(lane & 31) * 4;  // both lane halves fetch the same 32 scales
    }
    // (picked here once: picked per item, the two pointers become a table in scratch memory)
    const uint8_t *const x_src = (const uint8_t *)scalar_pointer(
        x_sums ? reinterpret_cast<const uint8_t *>(g.src.bs) : reinterpret_cast<const uint8_t *>(g.src.d));
    const uint8_t *f_x;
    const int8_t *f_q;
    const uint32_t lds_src = lds_address(lds + L::OFF_SRC);
    int w_last_row = -1;
    int w_ord = 0, w_kb = 0, w_step = 0, a_ord = 0, a_kb = 0, a_step = 0;
    constexpr int SLICES = 8 / L::RG, SLICE_STEP = GATHER ? 32 * L::RG : 1024 * L::RG;  // quant slices of a wavefront, their distance
    bool f_two = false;  // the activations' cursor's tile has rows in its second half
    auto weights_at = [&](const Item &it) {  // uniform
        const uint8_t *W = (it.mat ? g.W[1] : g.W[0]) + (size_t)it.expert * g.rows * g.row_stride;
        const int row_base = min(it.row_group * (32 * L::RG) + wave * 32, g.rows - 1), last_row = min(g.rows - 1 - row_base, 31);
        if (last_row != w_last_row) {  // (the offsets differ in a last partial row group only)
            w_last_row = last_row;
            wside.offsets((uint32_t)g.row_stride, last_row, lane);
            wside.pin();
        }
        wside.point_at(g, W, row_base, 0);
    };
    auto acts_at = [&](const Item &it, int ord) {  // uniform
        const int t = it.tile;
        f_two = it.count > 32;
        if (GATHER) {
            // piece (row, 16-byte half hk) of quant slice `wave`: bytes 32 * wave + 16 * hk of the row's block (SLICE_STEP on: the other slice's);
            // of the sums: 16 * hk of the block's 32 bytes; the scale: the block's 4 bytes
            uint32_t src;  // this lane's source rows of the tile (row lane % 32 of either half)
            asm volatile("ds_read_b32 %0, %1\n\ts_waitcnt lgkmcnt(0)" : "=v"(src) : "v"(lds_src + ord * 128 + (lane & 31) * 4));
            const uint32_t row_a = src & 0xffffu, row_b = src >> 16, hk = (uint32_t)(lane >> 5) * 16;
            const uint32_t cols = (uint32_t)nb * QK_K, row = x_second ? row_b : row_a;
            qa_off = row_a * cols + (uint32_t)wave * 32 + hk;
            qb_off = row_b * cols + (uint32_t)wave * 32 + hk;
            x_off = x_sums ? row * (uint32_t)nb * 32 + hk : row * (uint32_t)nb * 4;
            asm volatile("" : "+v"(qa_off), "+v"(qb_off), "+v"(x_off));
            f_q = g.src.q;
            f_x = x_src;
        } else {
            const size_t rec = (size_t)(2 * t + (x_second ? 1 : 0)) * nb;  // the small piece's half
            f_q = g.a.q + (size_t)2 * t * nb * 8192;
            f_x = x_sums ? reinterpret_cast<const uint8_t *>(g.a.bs + rec * 512)
                         : reinterpret_cast<const uint8_t *>(g.a.d + rec * 32);
        }
    };
    auto fetch_acts = [&]() {  // of the cursor's step; moves the cursor on
        const uint32_t st = lds_address(lds) + L::OFF_A + (uint32_t)(a_step & 1) * L::A_STAGE;
#pragma unroll
        for (int c = 0; c < SLICES; c++) dma16(st + (wave + c * L::RG) * 1024, f_q + c * SLICE_STEP, qa_off);
        if (f_two) {
#pragma unroll
            for (int c = 0; c < SLICES; c++) dma16(st + L::A_HALF + (wave + c * L::RG) * 1024, f_q + c * SLICE_STEP, qb_off);
        }
        if (x_small && (!x_second || f_two)) {
            const uint32_t half = st + (x_second ? L::A_HALF : 0);
            if (MINS && x_sums) dma16(half + L::A_BS, f_x, x_off);
            else dma4(half + L::A_DA, f_x, x_off);
        }
        f_q += GATHER ? QK_K : 8192;
        f_x += GATHER ? (x_sums ? 32 : 4) : (x_sums ? 1024 : 128);
        a_step++;
        if (++a_kb == nb) {
            a_kb = 0;
            if (++a_ord < my_items) acts_at(item(a_ord), a_ord);
        }
    };
    const uint32_t lds_w = lds_address(lds) + (uint32_t)wave * L::W_WAVE;
    auto fetch_weights = [&]() {  // of the cursor's step; moves the cursor on
        wside.fetch(lds_w + (uint32_t)(L::W_STAGES == 2 ? w_step & 1 : 0) * L::W_STAGE, lane);
        w_step++;
        if (++w_kb == nb) {
            w_kb = 0;
            if (++w_ord < my_items) weights_at(item(w_ord));
        } else {
            wside.move_on(w_kb - 1);
        }
    };
    // prologue: the activations of step 0, as many steps' weights as there are stages
    {
        const Item it = item(0);
        weights_at(it);
        acts_at(it, 0);
    }
    fetch_acts();
    fetch_weights();
    if (total_steps > 1 && L::W_STAGES > 1) fetch_weights();
    wait_vm<0>();
    lds_barrier();

    // ---- the arithmetic.  The unpacked weights are double-buffered in registers: while step s is
    // multiplied out of one set, step s+1 is unpacked into the other, the unpacking's vector
    // instructions filling the gaps between the MFMAs, each of which waits for the one before it.
    // (Every wavefront overlaps its own two kinds of work, so the wavefronts of a SIMD need not
    // be kept in different phases.)  The loop body exists twice, one copy per set. ----
    const uint32_t lds0 = lds_address(lds);
    BPlanes B0, B1;
    v16f accF0 = v16f{0.0f}, accF1 = v16f{0.0f};  // the tile's two halves
    const bool fetch_late = wave >= L::RG / 2;
    int c_ord = 0, c_kb = 0, c_step = 0;
    Item c_item = {0, 0, 0, 0, 0, 0};
    bool pending = false;  // `done` is an item whose results wait to be stored
    Item done = c_item;
    auto raw_of_step = [&](int s) {  // this lane's part of its row's block, read and arrived
        const int l = opaque_lane();
        typename Side::Raw R;
        Side::read(R, lds_w + (uint32_t)(L::W_STAGES == 2 ? s & 1 : 0) * L::W_STAGE, l & 31, l >> 5);
        return R;
    };
    auto multiply_half = [&](uint32_t st, v16f &accF, const BPlanes &B, auto between) {
        const int lane = opaque_lane(), lg = lane >> 5;
        TileOperands T;
        TileScales S;
        TileAcc X;
        read_ops<MINS>(T, st + lane * 16, st + L::A_BS + lane * 16);
        tile_mfmas_as_they_land<MINS, Side::SHIFT>(T, B, X, between);
        read_scales(S, st + L::A_DA + lg * 16);
        wait_scales<0>(S);
        tile_epilogue<MINS>(X, S, B, accF);
        // the epilogue must not sink below the next half's operand reads (its inputs would stay
        // live through that half's MFMAs): an empty volatile statement that "modifies" the sums
        // keeps its place among the volatile LDS reads
        asm volatile("" : "+v"(accF));
    };
    // (the next step's block R is unpacked into Bnext from inside the first half's chain of MFMAs)
    auto multiply_step = [&](const BPlanes &B, const typename Side::Raw &R, BPlanes &Bnext) {
        const uint32_t st = lds0 + L::OFF_A + (uint32_t)(c_step++ & 1) * L::A_STAGE;
        if (c_kb == 0) c_item = item(c_ord++);
        const int lg_next = opaque_lane() >> 5;
        const typename Side::Scales sc = Side::scales(R, lg_next);
        const int kb_next = c_kb + 1 == nb ? 0 : c_kb + 1;
        multiply_half(st, accF0, B, [&](int i, v16i &) { Side::unpack_piece(i, R, sc, lg_next, kb_next, Bnext); });
        if (c_item.count > 32) multiply_half(st + L::A_HALF, accF1, B, NothingBetween());
        if (++c_kb == nb) {
            pending = true;
            done = c_item;
            c_kb = 0;
        }
    };
    // a finished item's results are stored at the top of the next step: a store counts in vmcnt like
    // a load, and there it has the whole step before the wait at the step's end
    auto store_item = [&]() {  // a lane holds one weight row and 16 rows of the tile
        const int count = done.count;
        const int l = opaque_lane(), li = l & 31, lg = l >> 5;
        const int row = done.row_group * (32 * L::RG) + wave * 32 + li;
        int rows = g.rows;
        asm volatile("" : "+s"(rows));  // opaque: keeps the 16 row offsets from being hoisted out of the loop and held
        float *y = (done.mat ? g.y[1] : g.y[0]) + (size_t)done.y_row * rows;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int tok = (r >> 2) * 8 + lg * 4 + (r & 3);
            if (row < rows && tok < count) y[(uint32_t)(tok * rows + row)] = accF0[r];
        }
        accF0 = v16f{0.0f};
        if (count > 32) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const int tok = 32 + (r >> 2) * 8 + lg * 4 + (r & 3);
                if (row < rows && tok < count) y[(uint32_t)(tok * rows + row)] = accF1[r];
            }
            accF1 = v16f{0.0f};
        }
    };

    {  // step 0's weights into the first set; its stage is refilled at once
        const typename Side::Raw R = raw_of_step(0);
        const typename Side::Scales sc = Side::scales(R, lg);
#pragma unroll
        for (int i = 0; i < 9; i++) Side::unpack_piece(i, R, sc, lg, 0, B0);
        if (total_steps > L::W_STAGES) fetch_weights();
        if (L::W_STAGES == 1) wait_vm<0>();  // (step 1's, which step 0 unpacks)
    }
    auto step = [&](int s, const BPlanes &Bcur, BPlanes &Bnext) {
        if (pending) {
            store_item();
            pending = false;
        }
        // step s+1's raw weights leave LDS, which frees their stage (past the last step: whatever the stage holds,
        // unpacked into a set nobody will use)
        const typename Side::Raw R = raw_of_step(s + 1);
        // A wavefront is stalled while its loads wait for the CU's one address unit: half of a workgroup's wavefronts
        // fetch their weights before they multiply and half after, and the unit serves the one half while the other half
        // has the matrix cores.  The activations of the step behind this one are wanted at its end and go out first (into
        // the stage last read in step s-1).
        const bool more = s + 1 + L::W_STAGES < total_steps;
        if (s + 1 < total_steps) fetch_acts();
        if (more && !fetch_late) fetch_weights();
        multiply_step(Bcur, R, Bnext);
        if (more && fetch_late) fetch_weights();
        // What may be in flight past this wait: with two stages the weights of step s + 3, asked for in this step (the youngest loads
        // on either side of the products: the activations and a finished item's stores went out before them); step s + 1's activations
        // and step s + 2's weights, which step s + 1 unpacks, have landed.  With one stage (step s + 2's weights are the ones
        // just asked for), or where this step asked for none: nothing.  The barrier then makes the activations, fetched by four
        // wavefronts, everybody's, and the stage that this step read free.
        if (more && L::W_STAGES > 1) wait_vm<Side::REQUESTS>();
        else wait_vm<0>();
        lds_barrier();
    };
    for (int s = 0; s < total_steps; s += 2) {
        step(s, B0, B1);
        if (s + 1 < total_steps) step(s + 1, B1, B0);
    }
    if (pending) store_item();
}

template <bool GATHER>
__global__ __launch_bounds__(256, 2) void gemm_q4_k_stream_kernel(StreamArgs g) {
    stream_gemm<FRK_KIND_Q4_K, GATHER>(g);
}
__global__ __launch_bounds__(256, 2) void gemm_q6_k_stream_kernel(StreamArgs g) { stream_gemm<FRK_KIND_Q6_K, false>(g); }

// ------------------------------------------------------------------ launchers

#define FRK_LAUNCH_CHECK(what)                                                                          \
    do {                                                                                                \
        hipError_t e_ = hipGetLastError();                                                              \
        if (e_ != hipSuccess) return set_error(FRK_ERR_HIP, what " launch: %s", hipGetErrorString(e_)); \
    } while (0)

// ---- the tiled activations ----
static size_t tiled_records(size_t rows, size_t cols) { return (rows + 31) / 32 * (cols / QK_K); }
size_t q8k_tiled_bytes(size_t rows, size_t cols) {
    // the scales end with slack: a wavefront fetches 64 of them where 32 are used
    return tiled_records(rows, cols) * (8192 + 1024 + 128) + 256;
}
Q8KTiled q8k_tiled_carve(void *base, size_t rows, size_t cols) {
    const size_t rec = tiled_records(rows, cols);
    Q8KTiled a;
    a.q = (int8_t *)base;
    a.bs = (_Float16 *)((char *)base + rec * 8192);
    a.d = (float *)((char *)base + rec * (8192 + 1024));
    return a;
}
template <int WAVES>
static int launch_quantize_records(const float *x, size_t rows, size_t nb, const int *gather, size_t n_rec, Q8KTiled out,
                                   hipStream_t s, Q8KActsOut plain = Q8KActsOut()) {
    hipLaunchKernelGGL((quantize_q8_k_tiled_kernel<WAVES>), dim3((unsigned)n_rec), dim3(64 * WAVES), 0, s, x, (int)rows,
                       (int)nb, gather, out, plain);
    FRK_LAUNCH_CHECK("quantize_q8_k_tiled");
    return FRK_OK;
}
int launch_quantize_q8_k_tiled(const float *x, size_t rows, size_t cols, Q8KTiled out, hipStream_t s, Q8KActsOut plain) {
    const size_t nb = cols / QK_K, n_rec = (rows + 31) / 32 * nb;
    if (n_rec == 0) return FRK_OK;
    // Up to 400 records without LDS: a launch of 2.5 to 5 us is its chain of dependent steps, and a record's barrier and copies are the longer one;
    // past that both are bound by the stores, which a record's are the wider of.  us, launch after launch, a record / eight rows a workgroup: 48 x 4096
    // 3.08 / 2.49, 64 x 8192 3.12 / 2.41, 197 x 4096 3.22 / 2.54, 200 x 14336 5.27 / 4.92, 512 x 4096 3.75 / 3.72, but 512 x 14336
    // 8.79 / 8.92, 2000 x 8192 16.7 / 19.4, 2048 x 14336 28.5 / 33.6.
    if (n_rec <= 400) {
        hipLaunchKernelGGL(quantize_q8_k_octets_kernel, dim3((unsigned)(n_rec * 4)), dim3(512), 0, s, x, (int)rows, (int)nb, out, plain);
        FRK_LAUNCH_CHECK("quantize_q8_k_octets");
        return FRK_OK;
    }
    // (sixteen wavefronts a record, two rows each, at every size, us under the profiler, sixteen / eight / four: 512x4096 5.9 / 7.1 /
    // 10.2, 512x14336 10.4 / 12.0 / 14.0, 700x12288 10.6 / 12.0 / 13.5, 2000x8192 16.8 / 18.6 / 22.0)
    return launch_quantize_records<16>(x, rows, nb, nullptr, n_rec, out, s, plain);
}
// Q8_K rows as the quantizer of a thin batch leaves them, in the tiled form: a record a workgroup
__global__ __launch_bounds__(256) void tile_q8_k_kernel(Q8KActs a, int rows, int nb, Q8KTiled out) {
    const int t32 = blockIdx.x / nb, kb = blockIdx.x % nb;
    const size_t rec = (size_t)t32 * nb + kb;
    for (int i = threadIdx.x; i < 512; i += 256) {  // 16-byte piece: slice i / 64, half i / 32 % 2, row i % 32
        const int row = t32 * 32 + (i & 31);
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (row < rows) v = *reinterpret_cast<const uint4 *>(a.q + ((size_t)row * nb + kb) * QK_K + (i >> 6) * 32 + ((i >> 5) & 1) * 16);
        reinterpret_cast<uint4 *>(out.q + rec * 8192)[i] = v;
        const int sum_row = t32 * 32 + ((i >> 3) & 31), g = (i >> 8) * 8 + (i & 7);
        out.bs[rec * 512 + i] = sum_row < rows ? (_Float16)a.bsums[((size_t)sum_row * nb + kb) * 16 + g] : (_Float16)0.0f;
    }
    const int row = t32 * 32 + (int)threadIdx.x;
    if (threadIdx.x < 32) out.d[rec * 32 + threadIdx.x] = row < rows ? a.d[(size_t)row * nb + kb] : 0.0f;
}
int launch_tile_q8_k(const Q8KActs &a, size_t rows, size_t cols, Q8KTiled out, hipStream_t s) {
    const size_t nb = cols / QK_K, n_rec = (rows + 31) / 32 * nb;
    if (n_rec == 0) return FRK_OK;
    hipLaunchKernelGGL(tile_q8_k_kernel, dim3((unsigned)n_rec), dim3(256), 0, s, a, (int)rows, (int)nb, out);
    FRK_LAUNCH_CHECK("tile_q8_k");
    return FRK_OK;
}
int launch_quantize_q8_k_gather(const float *x, size_t cols, const int *gather, size_t max_rows, Q8KTiled out,
                                hipStream_t s) {
    const size_t nb = cols / QK_K, n_rec = max_rows / 32 * nb;
    if (n_rec == 0) return FRK_OK;
    return n_rec <= 1024 ? launch_quantize_records<16>(x, 0, nb, gather, n_rec, out, s)
                         : launch_quantize_records<4>(x, 0, nb, gather, n_rec, out, s);
}

// Which tile and split a batch takes: the one that an estimate of the launch's time finds cheapest.  A workgroup of the
// large tile (256 rows x 128 tokens) takes `step` microseconds per block of a row, one of the small tile (128 x 64) per two
// blocks -- longer, by `load`, the more of the 256 CUs have a workgroup (L2 and the clock are shared) -- and `start` for its
// first block and its stores; a launch is as many rounds of workgroups as the CUs take, which holds because every XCD has an
// equal share of them (deal_entry); splitting the blocks costs the second launch and its bytes.  The constants are a fit
// (4 % rms) to 6079 launches over 1200 drawn shapes: the three kinds, 1024 .. 14336 rows and columns, 8 .. 2048 tokens,
// 1 .. 8 parts.  Over the 720 of them with 48 tokens and more the choice is 0.2 % behind the best one measured on average,
// 8 % at worst; with the constants fitted to one half and tried on the other likewise.  (33 .. 64 tokens the small tile, the
// cheaper one there in every launch measured: its float step is the thin kernels', see fold_mins.)
// The last token tile of 128 multiplies only the 32-token tiles that have rows in use (three, two and one of four measured at 0.85, 0.7
// and 0.55 of a full block's time) and may be split into parts of its own number, so that its workgroups take about as long as the
// others: 197 tokens of 11008 x 4096 in Q5_K, three parts of the first tile and two of the second in one round of 215 workgroups,
// 47.9 -> 44.7 us.  Over 90 drawn shapes of 33 .. 2048 tokens whose plan these two change 0.92 of the time, 0.80 at best, 1.03 at
// worst.
PipePlan pipe_plan(int kind, size_t rows, size_t M, size_t nb) {
    struct Cost {
        float step, load, start;
    };
    // (a Q5_K or Q6_K block has three times Q4_K's vector instructions in its unpacking)
    const Cost small = kind == FRK_KIND_Q4_K ? Cost{1.62f, 0.74f, 3.26f} : Cost{2.41f, 0.77f, 4.06f};
    const Cost large = kind == FRK_KIND_Q4_K ? Cost{2.66f, 1.07f, 4.85f} : Cost{3.26f, 1.06f, 5.79f};
    auto rounds_us = [](size_t wgs, float steps, Cost c) {
        const float last = (float)(wgs % 256) / 256.0f;
        return (float)(wgs / 256) * (steps * (c.step + c.load) + c.start) + (wgs % 256 ? steps * (c.step + c.load * last) + c.start : 0.0f);
    };
    PipePlan best = {128, 64, 1, 1};
    float best_us = 0.0f;
    // Up to 32 tokens a tile of 64 rows x 32 tokens, four blocks a step: half the small tile's matrix instructions for the same
    // weights.  The same estimate, fitted (3.6 % rms) to 1700 launches over 130 shapes: its choice is 0.1 % behind the
    // best measured split on average and 3 % at worst.  With quantization, the small tile -> this one, us: Q4_K 14336x4096
    // at 9 and 32 rows 20.0 -> 14.9 and 21.6 -> 15.9, 4096x11008 at 16 20.0 -> 16.9, Q5_K 4096x4096 at 32 17.7 -> 14.4, Q6_K
    // 4096x11008 at 32 24.3 -> 21.3.
    if (M <= 32) {
        const Cost c = kind == FRK_KIND_Q4_K ? Cost{1.06f, 0.65f, 2.47f} : Cost{1.91f, 0.68f, 2.95f};
        best = {64, 32, 1, 1};
        for (int ks : {1, 2, 3, 4, 5, 6, 8, 12, 16}) {
            const size_t bytes = (size_t)ks * M * rows * sizeof(float);
            if (ks > 1 && (nb / (size_t)ks < 2 || bytes > SPLIT_PARTS_BYTES)) continue;
            const size_t wgs = (rows + 63) / 64 * (size_t)ks, blocks = (nb + (size_t)ks - 1) / (size_t)ks;
            const float us = rounds_us(wgs, (float)((blocks + 3) / 4), c) + (ks > 1 ? 1.6f + 2.6e-7f * (float)bytes : 0.0f);
            if (best_us == 0.0f || us < best_us) best_us = us, best.k_split = best.k_last = ks;
        }
        return best;
    }
    // First at a full price for every token tile, then, within that plan's tile, with the last token tile at its own. Neither
    // form of the choice is to cost precision.  2-norm against 64-bit sums, emulated with normal weights, rows of 32 blocks: the mins
    // folded (the large tile, see fold_mins) 1.4e-7 as one sum, 1.2e-7 in four; apart (the small tile, two sums a part) 9.7e-8
    // in two, 8.7e-8 in four; Q6_K 1.2e-7 as one sum, 1.0e-7 in two, 9.0e-8 in three, from five on 8.8e-8.  So the tile stays
    // (96 x 14336 x 8192 in Q4_K, tokens first, 42.4 us in the large one and 50.3 in the small one; Q6_K, whose error is the same in both, was
    // 0.95 to 1.04 of the time there), and no token tile's blocks are added up in fewer sums than before, or than five.
    // (Another plan than the first where it is ahead by 2 %: 222 x 11624 x 3328 in Q6_K, 1 % ahead by the estimate, 46.3 -> 47.9 us.)
    PipePlan full = best;
    for (int pass = 0; pass < 2; pass++) {
        best_us = 0.0f;
        for (int big = 0; big < (M > 64 ? 2 : 1); big++) {
            if (pass && (big ? 256 : 128) != full.rows_wg) continue;
            const Cost c = big ? large : small;
            const size_t row_tiles = big ? (rows + 255) / 256 : (rows + 127) / 128, tok_tiles = big ? (M + 127) / 128 : (M + 63) / 64;
            // the last token tile's 32-token tiles in use, and what a block of it costs of a full one's
            const size_t before = (tok_tiles - 1) * (big ? 128 : 64), in_use = (M - before + 31) / 32;
            const float share = !pass || !big || in_use == 4 ? 1.0f : in_use == 3 ? 0.85f : in_use == 2 ? 0.7f : 0.55f;
            for (int ks : {1, 2, 3, 4, 5, 6, 8})
                for (int last : {1, 2, 3, 4, 5, 6, 8}) {
                    const size_t wgs = row_tiles * ((tok_tiles - 1) * (size_t)ks + (size_t)last), most = (size_t)std::max(ks, last);
                    // (five parts, and other parts for the last token tile, where all workgroups are there at once)
                    if (last != ks && (!pass || !big || tok_tiles == 1 || in_use == 4)) continue;
                    if ((last != ks || ks == 5) && (!pass || wgs > 256)) continue;
                    if (most > 1 && (nb / most < 2 || most * M * rows * sizeof(float) > SPLIT_PARTS_BYTES)) continue;
                    const int shares = big ? 1 : 2;  // (of a part, in a workgroup)
                    if (pass && std::min(ks, last) * shares < std::min(full.k_split * shares, 5)) continue;
                    auto steps = [&](int parts) {
                        const size_t blocks = (nb + (size_t)parts - 1) / (size_t)parts;
                        return (float)(big ? blocks : (blocks + 1) / 2);
                    };
                    float us = rounds_us(wgs, steps(ks) * (tok_tiles == 1 ? share : 1.0f), c);
                    if (last != ks) {
                        const float step = c.step + c.load * (float)wgs / 256.0f;
                        us = std::max(steps(ks), steps(last) * share) * step + c.start;
                    }
                    if (most > 1) us += 1.3f + 2.6e-7f * (float)(((size_t)ks * before + (size_t)last * (M - before)) * rows * sizeof(float));
                    if (last != ks) us *= 1.03f;  // (the full tiles and the last one share no weights in an XCD's L2)
                    if (pass && (ks != full.k_split || last != ks)) us *= 1.02f;
                    if (best_us == 0.0f || us < best_us) {
                        best_us = us;
                        best = big ? PipePlan{256, 128, ks, last} : PipePlan{128, 64, ks, last};
                    }
                }
        }
        if (!pass) full = best;
    }
    return best;
}
size_t pipe_gemm_parts_bytes(int kind, size_t M, size_t cols, size_t rows) {
    const PipePlan p = pipe_plan(kind, rows, M, cols / QK_K);
    const size_t parts = (size_t)std::max(p.k_split, p.k_last);
    return parts > 1 ? parts * M * rows * sizeof(float) : 0;
}

int launch_pipe_gemm_acts(const frk_weights *w, Q8KTiled acts, size_t M, float *y, void *parts, hipStream_t s) {
    // the kernel addresses a row group's weights with 32-bit lane offsets
    if ((uint64_t)w->layout.row_stride * 64 >= (1ull << 32))
        return set_error(FRK_ERR_SHAPE, "matrix-core GEMM: rows of %zu bytes are beyond the kernel's offsets", w->layout.row_stride);
    const PipePlan p = pipe_plan(w->kind, w->rows, M, w->cols / QK_K);
    const GemmArgs g = pipe_args(w, acts, M, y, (float *)parts, p);
    if (w->kind == FRK_KIND_Q6_K) return launch_pipe_q6_k(g, p.rows_wg, s);
#define FRK_GO(KIND, KERNEL)                                                                                       \
    return p.rows_wg == 256   ? launch_pipe<KIND, 8, 1, 4>(KERNEL<8, 1, 4>, g, s)                                  \
           : p.rows_wg == 128 ? launch_pipe<KIND, 4, 2, 2>(KERNEL<4, 2, 2>, g, s) : launch_pipe<KIND, 2, 4, 1>(KERNEL<2, 4, 1>, g, s)
    if (w->kind == FRK_KIND_Q5_K) FRK_GO(FRK_KIND_Q5_K, gemm_q5_k_pipe_kernel);
    FRK_GO(FRK_KIND_Q4_K, gemm_q4_k_pipe_kernel);
#undef FRK_GO
}

template <int KIND, bool GATHER>
static int launch_stream(void (*kernel)(StreamArgs), const StreamArgs &g, int max_tiles, hipStream_t s) {
    using L = StreamLds<KIND, GATHER>;
    static int grid = 0;
    if (grid == 0) {
        int dev = 0, cus = 0;
        hipError_t e = hipGetDevice(&dev);
        if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
        if (e == hipSuccess) e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)L::BYTES);
        if (e != hipSuccess) return set_error(FRK_ERR_HIP, "grouped GEMM setup: %s", hipGetErrorString(e));
        grid = 2 * (cus < 8 ? 8 : cus / 8 * 8);  // two workgroups per CU, a multiple of the 8 XCDs
    }
    // more than two workgroups a CU (which then follow one another) when a workgroup's share of the largest possible list
    // would not fit its item table
    const size_t most_items = ((size_t)max_tiles + 7) / 8 * g.n_mat * g.row_tiles;
    const unsigned rounds = (unsigned)((most_items + (size_t)(grid / 8) * L::MAX_ITEMS - 1) /
                                       ((size_t)(grid / 8) * L::MAX_ITEMS));
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid * (rounds ? rounds : 1)), dim3(64 * L::RG), L::BYTES, s, g);
    FRK_LAUNCH_CHECK("grouped GEMM");
    return FRK_OK;
}

bool gemm_q4_k_stream_gathers(size_t src_rows, size_t cols) {
    // a source row is a 16-bit entry of the kernel's table, a row's place a 32-bit lane offset
    return src_rows <= 65535 && src_rows * cols < (1ull << 32);
}

int launch_gemm_k_stream(const frk_weights *w0, const frk_weights *w1, size_t rows_e, Q8KTiled a,
                            const Q8KRows *src, const int *gather, const int4 *tiles, const int *n_tiles,
                            int max_tiles, float *y0, float *y1, hipStream_t s) {
    if ((w0->kind != FRK_KIND_Q4_K && w0->kind != FRK_KIND_Q6_K) || (w1 && w1->kind != w0->kind))
        return set_error(FRK_ERR_UNSUPPORTED, "the grouped K-quant GEMM takes Q4_K or Q6_K stacks (kinds %d and %d)", w0->kind, w1 ? w1->kind : w0->kind);
    StreamArgs g;
    g.W[0] = w0->dev;
    g.W[1] = w1 ? w1->dev : w0->dev;
    g.y[0] = y0;
    g.y[1] = y1;
    g.n_mat = w1 ? 2 : 1;
    g.row_stride = w0->layout.row_stride;
    g.off_qh = (uint32_t)w0->layout.off_a;
    g.off_sc = (uint32_t)w0->layout.off_b;
    g.off_d = (uint32_t)w0->layout.off_c;
    g.rows = (int)rows_e;
    g.nb = (int)(w0->cols / QK_K);
    g.a = a;
    g.tiles = tiles;
    g.n_tiles = n_tiles;
    g.row_tiles = (int)((rows_e + 127) / 128);
    g.src = src ? *src : Q8KRows{nullptr, nullptr, nullptr};
    g.gather = gather;
    if (w0->kind == FRK_KIND_Q6_K) return launch_stream<FRK_KIND_Q6_K, false>(gemm_q6_k_stream_kernel, g, max_tiles, s);
    return src ? launch_stream<FRK_KIND_Q4_K, true>(gemm_q4_k_stream_kernel<true>, g, max_tiles, s)
               : launch_stream<FRK_KIND_Q4_K, false>(gemm_q4_k_stream_kernel<false>, g, max_tiles, s);
}

}  // namespace frk
