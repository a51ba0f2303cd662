// The pipelined matrix-core GEMM of the K-quants, shared by frk_gemm.hip (Q4_K, Q5_K) and frk_gemm_q6.hip (Q6_K):
// block layouts, the unpacking of a block into two int8 operand planes, and the kernel's body.
//
// A block's scaled codes go through int8 MFMAs as two planes H and L, so that one accumulator holds the block's exact
// integer sum: the H chain of MFMAs first, its sums shifted left, then the L chain.
//   Q4_K: sc * q with sc = 8 * sh + sl: H = sh * q, L = sl * q (bytes below 106), a shift by 3.
//   Q5_K: p = sc * q (0 .. 1953) and Q6_K: p = sc * (q - 32) (-4064 .. 4096) are 16-bit numbers: H is the high byte of
//         p + 128, L the low byte of p as a signed number, p = 256 * H + L, a shift by 8.  The products are packed
//         16-bit multiply-adds and the bytes are picked by v_perm.
// (Before, Q5_K had a third plane for its fifth bits and Q6_K four planes, its scale and its code split in two each: 24
// and 32 MFMAs a tile and block where two planes take 16, and no registers left for the 256 x 128 tile.  M = 512, kernel
// alone: 14336x4096 in Q5_K 131 -> 78 us, 4096x14336 in Q6_K 155 -> 83 us with the sum of its four parts.)
#pragma once

#include "frk_deal.hpp"
#include "frk_device.hpp"

#include <type_traits>

namespace frk {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef unsigned short us2 __attribute__((ext_vector_type(2)));

struct GemmArgs {
    const uint8_t *W;
    size_t row_stride;
    uint32_t off_qh, off_sc, off_d;  // the planes of a Q6_K row
    int rows, nb, M;
    Q8KTiled a;  // ceil(M / 32) tiles
    float *y;    // [M][rows]
    int row_tiles, tok_tiles;
    int k_split;     // parts of a row's blocks; with more than one each writes its sums to `partial`
    int k_last;      // the parts of the last token tile
    float *partial;  // [k_split][M][rows], added up afterwards (launch_sum_parts)
    int parts_inner; // a row tile's parts next to each other in the work list
};

// One block of a lane's weight row as MFMA B operands: the two pre-scaled planes of the 8 sub-blocks,
// the mins as f16 and the block's two f32 scales.  (Named members, not arrays: they must stay in
// registers.)
struct BPlanes {
    v4i H0, H1, H2, H3, H4, H5, H6, H7;
    v4i L0, L1, L2, L3, L4, L5, L6, L7;
    v8h m;
    float d, ndmin;
};
struct RawBlock {  // header + the lane's 16-byte half of each 32-byte nibble pair, as read from LDS
    v4i wh, q0, q1, q2, q3;
};
// Q5_K: the same block with a fifth bit per weight -- byte l of the 32 bytes behind the header holds weight l of
// every sub-block, sub-block j in bit j (dot_q5_k_q8, crates/frink-quant/src/lib.rs:886-938); fh is the lane's
// 16-byte half of them.
struct RawBlock5 {
    v4i wh, q0, q1, q2, q3, fh;
};
// Q6_K, from the resident planar rows (layout_for): sub-blocks 4n .. 4n+3 are the weights 128n + 32J + 16lg + (0..15) --
// a nibble of l<n>a (J = 0, 2) or l<n>b (J = 1, 3), low nibbles for J = 0, 1, under two bits of h<n> (bits 2J..).
struct RawBlock6 {
    v4i l0a, l0b, l1a, l1b, h0, h1;
    v4i sc;  // the block's sixteen scales
    int d2;  // the f16 super-scales of this block and of its even or odd neighbour
};
struct TileOperands {  // one 32-token tile of a block: 8 k-slices of quants and the bsums
    v4i a0, a1, a2, a3, a4, a5, a6, a7;
    v8h bs;
};
struct TileScales {  // the tile's 16 block scales this lane's results need
    v4f da0, da1, da2, da3;
};

// LDS reads are issued from inline assembly so that the compiler's wait-count insertion does not see
// them: it cannot tell that an LDS read does not alias a stage a global_load_lds is still filling
// and would wait for vmcnt(0), i.e. for the whole prefetch, in front of every read.  The price is
// that the waits are placed by hand.  LDS operations of a wavefront complete in order, so
// "at most N outstanding" means everything but the N youngest reads has arrived; each wait names the
// registers it releases so that their uses cannot be scheduled above it.
#define FRK_DS_READ(dst, addr, off) asm volatile("ds_read_b128 %0, %1 offset:" #off : "=v"(dst) : "v"(addr))

__device__ __forceinline__ void read_raw(RawBlock &R, uint32_t header, uint32_t quants) {
    FRK_DS_READ(R.wh, header, 0);
    FRK_DS_READ(R.q0, quants, 16);
    FRK_DS_READ(R.q1, quants, 48);
    FRK_DS_READ(R.q2, quants, 80);
    FRK_DS_READ(R.q3, quants, 112);
}
// result register r belongs to token 8*(r/4) + 4*(lane/32) + r%4 of the tile
__device__ __forceinline__ void read_scales(TileScales &S, uint32_t scales) {
    FRK_DS_READ(S.da0, scales, 0);
    FRK_DS_READ(S.da1, scales, 32);
    FRK_DS_READ(S.da2, scales, 64);
    FRK_DS_READ(S.da3, scales, 96);
}
template <int N>
__device__ __forceinline__ void wait_scales(TileScales &S) {
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(S.da0), "+v"(S.da1), "+v"(S.da2), "+v"(S.da3) : "n"(N));
}
template <int N>
__device__ __forceinline__ void wait_raw(RawBlock &R) {
    asm volatile("s_waitcnt lgkmcnt(%5)" : "+v"(R.wh), "+v"(R.q0), "+v"(R.q1), "+v"(R.q2), "+v"(R.q3) : "n"(N));
}
template <int N>
__device__ __forceinline__ void wait_raw(RawBlock5 &R) {
    asm volatile("s_waitcnt lgkmcnt(%6)" : "+v"(R.wh), "+v"(R.q0), "+v"(R.q1), "+v"(R.q2), "+v"(R.q3), "+v"(R.fh) : "n"(N));
}
template <int N>
__device__ __forceinline__ void wait_raw(RawBlock6 &R) {
    asm volatile("s_waitcnt lgkmcnt(%8)"
                 : "+v"(R.l0a), "+v"(R.l0b), "+v"(R.l1a), "+v"(R.l1b), "+v"(R.h0), "+v"(R.h1), "+v"(R.sc), "+v"(R.d2)
                 : "n"(N));
}
template <int N>
__device__ __forceinline__ void wait_vm() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// The header of a Q4_K or Q5_K block: its 6-bit scales and mins.
struct BlockScales {
    uint32_t sc_lo, sc_hi, m_lo, m_hi;  // a byte per sub-block: 0..3 and 4..7
};
__device__ __forceinline__ BlockScales block_scales(const v4i &wh) {
    const uint32_t hy = (uint32_t)wh.y, hz = (uint32_t)wh.z, hw = (uint32_t)wh.w;
    BlockScales s;
    s.sc_lo = hy & 0x3f3f3f3fu;
    s.m_lo = hz & 0x3f3f3f3fu;
    s.sc_hi = (hw & 0x0f0f0f0fu) | (((hy >> 6) & 0x03030303u) << 4);
    s.m_hi = ((hw >> 4) & 0x0f0f0f0fu) | (((hz >> 6) & 0x03030303u) << 4);
    return s;
}
// lg = lane / 32 selects which half of every sub-block this lane holds
__device__ __forceinline__ void unpack_rest(const v4i &wh, const BlockScales &s, int lg, BPlanes &B) {
    // mins of the four sub-blocks whose 16-wide groups are 8*lg .. 8*lg+7, each twice
    const uint32_t hx = (uint32_t)wh.x;
    const uint32_t mw = lg ? s.m_hi : s.m_lo;
    const _Float16 m0 = (_Float16)(int)(mw & 0xff), m1 = (_Float16)(int)((mw >> 8) & 0xff);
    const _Float16 m2 = (_Float16)(int)((mw >> 16) & 0xff), m3 = (_Float16)(int)(mw >> 24);
    B.m = v8h{m0, m0, m1, m1, m2, m2, m3, m3};
    B.d = h2f(hx & 0xffffu);
    B.ndmin = -h2f(hx >> 16);
}

// The large tile's form of the float step, one accumulator less (there are no registers for it): the mins' MFMA
// adds onto the converted integer sums instead of into registers of its own.  With d' = d / (-dmin):
//     d * S1 - dmin * S2 = (-dmin) * (d' * S1 + S2),
// so the f16 MFMA takes d' * S1 as its C operand and the epilogue multiplies by -dmin (and the token's
// scale).  A row whose dmin is zero keeps d and a factor of one, and zero mins.  (Two roundings a block more than the
// two-term form of the small tile, which every batch of up to 64 rows takes, and of the thin kernels: 2-norm against
// 64-bit sums at 15 rows of Q4_K 2009x12032 1.3e-7 folded, 9.0e-8 apart, 9.2e-8 on the thin kernels; Q5_K 3594x8192 at 25
// 1.3e-7, 9.2e-8 and 9.0e-8.  In time the small tile's two forms are within 1 % of each other.)
__device__ __forceinline__ void fold_mins(BPlanes &B) {
    const bool z = B.ndmin == 0.0f;
    B.d = z ? B.d : B.d * __builtin_amdgcn_rcpf(B.ndmin);
    B.ndmin = z ? 1.0f : B.ndmin;
    if (z) B.m = v8h{0, 0, 0, 0, 0, 0, 0, 0};
}

// The block's scales as the packed multiply wants them: for sub-block j one register with sh_j = sc_j >> 3 in
// its low half and sl_j = sc_j & 7 in its high half.  The multiply picks a half for both of its 16-bit lanes
// through op_sel, so nothing has to be replicated.
struct ScalePairs {
    uint32_t p0, p1, p2, p3, p4, p5, p6, p7;
};
__device__ __forceinline__ ScalePairs scale_pairs(const BlockScales &s) {
    const uint32_t sh_lo = (s.sc_lo >> 3) & 0x07070707u, sl_lo = s.sc_lo & 0x07070707u;
    const uint32_t sh_hi = (s.sc_hi >> 3) & 0x07070707u, sl_hi = s.sc_hi & 0x07070707u;
    // v_perm_b32: selector bytes 0..3 take the second operand's bytes, 4..7 the first's, 0x0c gives zero
    ScalePairs r;
    r.p0 = __builtin_amdgcn_perm(sl_lo, sh_lo, 0x0c040c00u);
    r.p1 = __builtin_amdgcn_perm(sl_lo, sh_lo, 0x0c050c01u);
    r.p2 = __builtin_amdgcn_perm(sl_lo, sh_lo, 0x0c060c02u);
    r.p3 = __builtin_amdgcn_perm(sl_lo, sh_lo, 0x0c070c03u);
    r.p4 = __builtin_amdgcn_perm(sl_hi, sh_hi, 0x0c040c00u);
    r.p5 = __builtin_amdgcn_perm(sl_hi, sh_hi, 0x0c050c01u);
    r.p6 = __builtin_amdgcn_perm(sl_hi, sh_hi, 0x0c060c02u);
    r.p7 = __builtin_amdgcn_perm(sl_hi, sh_hi, 0x0c070c03u);
    return r;
}
// bytes of `nib` (each below 16) times the low (H) and the high (L) half of `pair`: bytes stay below 106
__device__ __forceinline__ void scaled_planes(uint32_t nib, uint32_t pair, int &h, int &l) {
    asm("v_pk_mul_lo_u16 %0, %1, %2 op_sel_hi:[1,0]" : "=v"(h) : "v"(nib), "v"(pair));
    asm("v_pk_mul_lo_u16 %0, %1, %2 op_sel:[0,1] op_sel_hi:[1,1]" : "=v"(l) : "v"(nib), "v"(pair));
}
__device__ __forceinline__ void unpack_pair_sel(const v4i q, uint32_t pair0, uint32_t pair1, v4i &H0, v4i &L0, v4i &H1, v4i &L1) {
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const uint32_t w = (uint32_t)q[c];
        int h0, l0, h1, l1;
        scaled_planes(w & 0x0f0f0f0fu, pair0, h0, l0);
        scaled_planes((w >> 4) & 0x0f0f0f0fu, pair1, h1, l1);
        H0[c] = h0, L0[c] = l0, H1[c] = h1, L1[c] = l1;
    }
}
// The same in plain vector arithmetic (the compiler finds the op_sel forms itself), for a kernel that leaves
// the place of the unpacking to the compiler: statements of inline assembly stay where they are written.
__device__ __forceinline__ void unpack_pair_free(const v4i q, uint32_t pair0, uint32_t pair1, v4i &H0, v4i &L0, v4i &H1, v4i &L1) {
    us2 p0, p1;
    __builtin_memcpy(&p0, &pair0, 4);
    __builtin_memcpy(&p1, &pair1, 4);
    const us2 h0 = {p0.x, p0.x}, l0 = {p0.y, p0.y}, h1 = {p1.x, p1.x}, l1 = {p1.y, p1.y};
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const uint32_t w = (uint32_t)q[c];
        const uint32_t nl = w & 0x0f0f0f0fu, nh = (w >> 4) & 0x0f0f0f0fu;
        us2 a, b;
        __builtin_memcpy(&a, &nl, 4);
        __builtin_memcpy(&b, &nh, 4);
        const us2 r0 = a * h0, r1 = a * l0, r2 = b * h1, r3 = b * l1;  // bytes stay below 106
        int o0, o1, o2, o3;
        __builtin_memcpy(&o0, &r0, 4);
        __builtin_memcpy(&o1, &r1, 4);
        __builtin_memcpy(&o2, &r2, 4);
        __builtin_memcpy(&o3, &r3, 4);
        H0[c] = o0, L0[c] = o1, H1[c] = o2, L1[c] = o3;
    }
}
__device__ __forceinline__ void unpack_block(const RawBlock &R, int lg, BPlanes &B) {
    const BlockScales s = block_scales(R.wh);
    const ScalePairs p = scale_pairs(s);
    unpack_pair_sel(R.q0, p.p0, p.p1, B.H0, B.L0, B.H1, B.L1);
    unpack_pair_sel(R.q1, p.p2, p.p3, B.H2, B.L2, B.H3, B.L3);
    unpack_pair_sel(R.q2, p.p4, p.p5, B.H4, B.L4, B.H5, B.L5);
    unpack_pair_sel(R.q3, p.p6, p.p7, B.H6, B.L6, B.H7, B.L7);
    unpack_rest(R.wh, s, lg, B);
}

// Four codes of one sub-block (a byte each) times a scale, plus a bias, as the two byte planes: with
// p' = code * scale + bias (16 bits, two's complement), where bias carries 128 (and Q6_K's -32 * scale), the high
// bytes are H and the low bytes less 128 are L.  The scale and the bias are the low halves of their registers.
__device__ __forceinline__ void byte_planes(uint32_t codes, uint32_t scale, uint32_t bias, int &h, int &l) {
    const uint32_t even = codes & 0x00ff00ffu, odd = __builtin_amdgcn_perm(0u, codes, 0x0c030c01u);
    const us2 s = {(unsigned short)scale, (unsigned short)scale}, b = {(unsigned short)bias, (unsigned short)bias};
    auto mad = [&](uint32_t v) {
        us2 c;
        __builtin_memcpy(&c, &v, 4);
        const us2 r = c * s + b;
        uint32_t out;
        __builtin_memcpy(&out, &r, 4);
        return out;
    };
    const uint32_t pe = mad(even), po = mad(odd);
    h = (int)__builtin_amdgcn_perm(po, pe, 0x07030501u);
    l = (int)(__builtin_amdgcn_perm(po, pe, 0x06020400u) ^ 0x80808080u);
}

template <int BY>
__device__ __forceinline__ uint32_t moved_up(uint32_t v) {  // by BY bits (down where BY is negative)
    if constexpr (BY >= 0) return v << BY;
    else return v >> -BY;
}
// Q5_K: a nibble pair's 16 bytes under the fifth bits of sub-blocks J and J + 1
template <int J>
__device__ __forceinline__ uint32_t fifth_over_nibbles(uint32_t fifth) {  // bit J of every byte as bit 4
    return moved_up<4 - J>(fifth) & 0x10101010u;
}
template <int J>
__device__ __forceinline__ void unpack_pair5(const v4i q, const v4i fh, uint32_t s0, uint32_t s1, v4i &H0, v4i &L0, v4i &H1, v4i &L1) {
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const uint32_t w = (uint32_t)q[c], f = (uint32_t)fh[c];
        int h0, l0, h1, l1;
        byte_planes((w & 0x0f0f0f0fu) | fifth_over_nibbles<J>(f), s0, 128u, h0, l0);
        byte_planes(((w >> 4) & 0x0f0f0f0fu) | fifth_over_nibbles<J + 1>(f), s1, 128u, h1, l1);
        H0[c] = h0, L0[c] = l0, H1[c] = h1, L1[c] = l1;
    }
}
__device__ __forceinline__ void unpack_block(const RawBlock5 &R, int lg, BPlanes &B) {
    const BlockScales s = block_scales(R.wh);
    const uint32_t lo = s.sc_lo, hi = s.sc_hi;
    auto scale = [](uint32_t four, int j) { return (four >> (8 * j)) & 0xffu; };
    unpack_pair5<0>(R.q0, R.fh, scale(lo, 0), scale(lo, 1), B.H0, B.L0, B.H1, B.L1);
    unpack_pair5<2>(R.q1, R.fh, scale(lo, 2), scale(lo, 3), B.H2, B.L2, B.H3, B.L3);
    unpack_pair5<4>(R.q2, R.fh, scale(hi, 0), scale(hi, 1), B.H4, B.L4, B.H5, B.L5);
    unpack_pair5<6>(R.q3, R.fh, scale(hi, 2), scale(hi, 3), B.H6, B.L6, B.H7, B.L7);
    unpack_rest(R.wh, s, lg, B);
}

// Q6_K: one sub-block of a half (J = 0..3), its nibbles out of `nib`, two more bits of each code out of `two`;
// `scales` holds the scales of this lane's two groups of sub-blocks J & ~1 and J | 1 in bytes 0 and 2.
template <int J>
__device__ __forceinline__ void unpack_sub6(const v4i nib, const v4i two, uint32_t scales, v4i &H, v4i &L) {
    const int s = (int)(int8_t)((J & 1) ? scales >> 16 : scales);
    const uint32_t bias = (uint32_t)(128 - 32 * s);
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const uint32_t n = (uint32_t)nib[c], t = (uint32_t)two[c];
        const uint32_t low = (J < 2 ? n : n >> 4) & 0x0f0f0f0fu;
        const uint32_t high = moved_up<4 - 2 * J>(t) & 0x30303030u;
        int h, l;
        byte_planes(low | high, (uint32_t)s, bias, h, l);
        H[c] = h, L[c] = l;
    }
}
template <int OFF>
__device__ __forceinline__ void ds_read16(v4i &dst, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF>
__device__ __forceinline__ void ds_read16(v8h &dst, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
template <int OFF>
__device__ __forceinline__ void ds_read16(v4f &dst, uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(dst) : "v"(addr), "n"(OFF));
}
// tile slot SLOT of a stage: its eight k-slices and (SUMS) its sums, in this order
template <int SLOT, bool SUMS>
__device__ __forceinline__ void read_tile(TileOperands &T, uint32_t qa, uint32_t ba) {
    ds_read16<SLOT * 8192 + 0>(T.a0, qa);
    ds_read16<SLOT * 8192 + 1024>(T.a1, qa);
    ds_read16<SLOT * 8192 + 2048>(T.a2, qa);
    ds_read16<SLOT * 8192 + 3072>(T.a3, qa);
    ds_read16<SLOT * 8192 + 4096>(T.a4, qa);
    ds_read16<SLOT * 8192 + 5120>(T.a5, qa);
    ds_read16<SLOT * 8192 + 6144>(T.a6, qa);
    ds_read16<SLOT * 8192 + 7168>(T.a7, qa);
    if (SUMS) ds_read16<SLOT * 1024>(T.bs, ba);
}
// operand J (0..7) of tile slot SLOT
template <int SLOT, int J>
__device__ __forceinline__ void read_tile_operand(TileOperands &T, uint32_t qa) {
    v4i &dst = J == 0 ? T.a0 : J == 1 ? T.a1 : J == 2 ? T.a2 : J == 3 ? T.a3 : J == 4 ? T.a4 : J == 5 ? T.a5 : J == 6 ? T.a6 : T.a7;
    ds_read16<SLOT * 8192 + J * 1024>(dst, qa);
}
template <int SLOT>
__device__ __forceinline__ void read_tile_sums(TileOperands &T, uint32_t ba) {
    ds_read16<SLOT * 1024>(T.bs, ba);
}
template <int SLOT>
__device__ __forceinline__ void read_tile_scales(TileScales &S, uint32_t sa) {
    ds_read16<SLOT * 128 + 0>(S.da0, sa);
    ds_read16<SLOT * 128 + 32>(S.da1, sa);
    ds_read16<SLOT * 128 + 64>(S.da2, sa);
    ds_read16<SLOT * 128 + 96>(S.da3, sa);
}

// A finished tile's way into the float sums, in sixteen pieces.  MINS_FOLDED (the arithmetic fold_mins prepares):
//   pieces 0..7   c[r] = d' * float(S1[r]) for two results each,
//   piece  7      then the mins' MFMA adds S2 onto c,
//   pieces 8..15  sum[r] += (da[r] * -dmin) * c[r] for two results each.
// MINS_APART: piece 0 S2 into registers of its own, pieces 0..7 c[r] = d * float(S1[r]), pieces 8..15
// sum[r] += da[r] * (c[r] - dmin * S2[r]).
// NO_MINS: c[r] = float(S1[r]), then sum[r] += (da[r] * d) * c[r].
enum { NO_MINS, MINS_FOLDED, MINS_APART };
struct TileTail {
    v16i s1;      // the integer sums
    v16f c;       // see above
    v16f s2;      // MINS_APART
    v8h bs;       // the tile's 16-wide activation sums
    TileScales S; // the tile's activation scales
};
template <int FORM>
__device__ __forceinline__ void tail_piece(int i, TileTail &E, const BPlanes &B, v16f &sum) {
    if (i < 8) {
        if (FORM == MINS_APART && i == 0) E.s2 = __builtin_amdgcn_mfma_f32_32x32x16_f16(E.bs, B.m, v16f{0.0f}, 0, 0, 0);
        E.c[2 * i] = FORM != NO_MINS ? B.d * (float)E.s1[2 * i] : (float)E.s1[2 * i];
        E.c[2 * i + 1] = FORM != NO_MINS ? B.d * (float)E.s1[2 * i + 1] : (float)E.s1[2 * i + 1];
        if (FORM == MINS_FOLDED && i == 7) E.c = __builtin_amdgcn_mfma_f32_32x32x16_f16(E.bs, B.m, E.c, 0, 0, 0);
    } else {
        const v4f dav[4] = {E.S.da0, E.S.da1, E.S.da2, E.S.da3};
        const float d = FORM == MINS_FOLDED ? B.ndmin : B.d;
#pragma unroll
        for (int r = 2 * (i - 8); r < 2 * (i - 8) + 2; r++) {
            if (FORM == MINS_APART) sum[r] = fmaf(dav[r >> 2][r & 3], fmaf(B.ndmin, E.s2[r], E.c[r]), sum[r]);
            else sum[r] = fmaf(dav[r >> 2][r & 3] * d, E.c[r], sum[r]);
        }
    }
}

// Up to four pieces of 1 KB that lie 1 KB apart in LDS and whose lane offsets already carry the matching
// distance in global memory: a request's instruction offset moves BOTH of its addresses (checked on the
// device), so one write of M0 serves the four.  `lds_uniform` and `base_uniform` must be scalar values.
template <int N>
__device__ __forceinline__ void dma16_run(uint32_t lds_uniform, const void *base_uniform, uint32_t o0, uint32_t o1, uint32_t o2,
                                          uint32_t o3) {
    static_assert(N >= 1 && N <= 4, "the instruction offset reaches 3072");
    if (N == 4)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %5\n\tglobal_load_lds_dwordx4 %2, %5 offset:1024\n\t"
                     "global_load_lds_dwordx4 %3, %5 offset:2048\n\tglobal_load_lds_dwordx4 %4, %5 offset:3072"
                     :
                     : "s"(lds_uniform), "v"(o0), "v"(o1), "v"(o2), "v"(o3), "s"(base_uniform)
                     : "memory");
    else if (N == 2)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %3\n\tglobal_load_lds_dwordx4 %2, %3 offset:1024"
                     :
                     : "s"(lds_uniform), "v"(o0), "v"(o1), "s"(base_uniform)
                     : "memory");
    else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_uniform), "v"(o0), "s"(base_uniform) : "memory");
}

// The sixteen integer MFMAs of a tile, its operands released two at a time: they were requested in the order a0..a7
// and then LATER more LDS reads (the tile's sums, the scales of the tile before).  between(i) runs after MFMA i has been
// issued; from MFMA 8 on operand a(i-8) has been read for the last time, and next(i-8) may request the next tile's into
// its place.
template <int N, class V>
__device__ __forceinline__ void wait_lgkm2(V &r0, V &r1, v16i &acc) {
    asm volatile("s_waitcnt lgkmcnt(%3)" : "+v"(r0), "+v"(r1), "+v"(acc) : "n"(N));
}
template <int LATER, bool SUMS, int SHIFT, class Between, class Next>
__device__ __forceinline__ v16i tile_chain(TileOperands &T, const BPlanes &B, Between between, Next next) {
    const v16i zi = {0};
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(T.a0), "+v"(T.a1) : "n"(6 + LATER));
    v16i acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a0, B.H0, zi, 0, 0, 0);
    between(0);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a1, B.H1, acc, 0, 0, 0);
    between(1);
    wait_lgkm2<4 + LATER>(T.a2, T.a3, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a2, B.H2, acc, 0, 0, 0);
    between(2);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a3, B.H3, acc, 0, 0, 0);
    between(3);
    wait_lgkm2<2 + LATER>(T.a4, T.a5, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a4, B.H4, acc, 0, 0, 0);
    between(4);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a5, B.H5, acc, 0, 0, 0);
    between(5);
    wait_lgkm2<LATER>(T.a6, T.a7, acc);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a6, B.H6, acc, 0, 0, 0);
    between(6);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a7, B.H7, acc, 0, 0, 0);
    between(7);
    if constexpr (SUMS) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(T.bs), "+v"(acc));  // (and the reads behind the sums)
    else asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(acc));
    acc = acc << SHIFT;
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a0, B.L0, acc, 0, 0, 0);
    between(8);
    next(0);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a1, B.L1, acc, 0, 0, 0);
    next(1);
    between(9);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a2, B.L2, acc, 0, 0, 0);
    next(2);
    between(10);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a3, B.L3, acc, 0, 0, 0);
    next(3);
    between(11);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a4, B.L4, acc, 0, 0, 0);
    next(4);
    between(12);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a5, B.L5, acc, 0, 0, 0);
    next(5);
    between(13);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a6, B.L6, acc, 0, 0, 0);
    next(6);
    between(14);
    acc = __builtin_amdgcn_mfma_i32_32x32x32_i8(T.a7, B.L7, acc, 0, 0, 0);
    next(7);
    between(15);
    return acc;
}

// ---------------------------------------------------------------------------------------------
// The dense kernel in its pipelined form.
//
// What bounds a SIMD here is its one issue port, not the matrix core alone: measured on this part, a
// v_mfma_i32_32x32x32_i8 keeps the matrix core 32 clocks but costs the SIMD about 20 clocks in which no
// vector instruction issues, and every vector instruction another 2.6 -- whichever wavefront they come
// from.  About five vector instructions fit between two MFMAs for free; a tile (16 + 1 MFMAs) has ~80
// of epilogue.  So the epilogue of tile t-1 is cut into sixteen pieces that ride in the gaps of tile
// t's chain of MFMAs, the address arithmetic of the prefetch is scalar (global_load_lds with a scalar
// base and lane offsets that are computed once), and what stays exposed is the unpacking of the
// next block and the last tile's epilogue.
//
// A workgroup = 8 wavefronts = RG row groups of 32 weight rows x KS shares of the blocks; a wavefront
// runs MT 32-token tiles against its rows' current block.  KS = 2 (small matrices: 128 rows x 64 tokens
// per workgroup fill the chip where 256 x 128 would not) and KS = 4 (64 rows x 32 tokens) share the blocks
// between wavefronts whose sums are added through LDS at the end, four of them as (0 + 1) + (2 + 3).
//
// LDS: activations in a ring of 3 stages (requested two steps ahead), their scales in a ring of 4
// (they are read by an epilogue that may run a step later), the raw weights in ONE slot per
// wavefront: a block leaves its slot for registers at the end of the step before it is multiplied,
// and the slot is refilled at once.  One barrier per step.
// ---- the weight side, by kind: how a wavefront's 32 rows of one block come into its LDS slot (piece by piece, at
// scalar pointers that move on by one block a request plus lane offsets that never change), leave it for registers, and
// become operand planes.  Rows past the matrix read its last row.  Requests that ride on another's M0 with an
// instruction offset have it move the global address too: their lane offsets are short of it by as much (the pointers
// are kept 4096 bytes low and the offsets 4096 high, so that none goes negative). ----
template <int KIND>
struct WeightSide {  // Q4_K, Q5_K: the rows' 9 or 11 sixteen-byte pieces back to back, piece 64 * c + lane in request c
    static constexpr bool Q5 = KIND == FRK_KIND_Q5_K;
    static constexpr int BB = Q5 ? Q5_K_BYTES : Q4_K_BYTES, PR = BB / 16;  // bytes of a block, its pieces
    static constexpr int NC = (32 * PR + 63) / 64;                         // requests (the last: half)
    static_assert(32 * PR == 64 * (NC - 1) + 32, "the last request of a block is 32 lanes wide");
    static_assert(NC == 5 || NC == 6, "four requests share one write of M0, the rest follow");
    static constexpr int SLOT = 32 * BB, SHIFT = Q5 ? 8 : 3, REQUESTS = NC;
    static constexpr bool MINS = true;
    using Raw = std::conditional_t<Q5, RawBlock5, RawBlock>;
    uint32_t off[NC];
    const uint8_t *src;
    __device__ __forceinline__ void offsets(uint32_t stride, int last_row, int lane) {  // rows past `last_row` (of 32) read it
#pragma unroll
        for (int c = 0; c < NC; c++) {
            const int p = 64 * c + lane;
            const int r = min(p / PR, last_row);
            off[c] = (uint32_t)r * stride + (uint32_t)(p % PR) * 16 + 4096u - (c < 4 ? 1024u * c : 0u);
        }
    }
    template <class Args>
    __device__ __forceinline__ void point_at(const Args &g, const uint8_t *W, int row_base, int kb) {
        src = (const uint8_t *)scalar_pointer(W + (size_t)row_base * g.row_stride + (size_t)kb * BB - 4096);
    }
    __device__ __forceinline__ void fetch(uint32_t slot, int lane) {
        dma16_run<4>(slot, src, off[0], off[1], off[2], off[3]);
        if (NC == 6) dma16_run<1>(slot + 4096, src, off[4], 0, 0, 0);
        if (lane < 32) dma16_run<1>(slot + (NC - 1) * 1024, src, off[NC - 1], 0, 0, 0);
    }
    __device__ __forceinline__ void move_on(int) { src += BB; }
    static __device__ __forceinline__ void read(Raw &R, uint32_t slot, int li, int lg) {
        const uint32_t wa = slot + li * BB;
        if constexpr (Q5) {  // (the nibbles sit behind the 32 bytes of fifth bits)
            FRK_DS_READ(R.fh, wa + 16 * lg, 16);
            FRK_DS_READ(R.wh, wa, 0);
            FRK_DS_READ(R.q0, wa + 16 * lg, 48);
            FRK_DS_READ(R.q1, wa + 16 * lg, 80);
            FRK_DS_READ(R.q2, wa + 16 * lg, 112);
            FRK_DS_READ(R.q3, wa + 16 * lg, 144);
        } else {
            read_raw(R, wa, wa + 16 * lg);
        }
        wait_raw<0>(R);
    }
    static __device__ __forceinline__ void unpack(const Raw &R, int lg, int, BPlanes &B) { unpack_block(R, lg, B); }
    __device__ __forceinline__ void pin() {  // the lane offsets stay in registers as they are
#pragma unroll
        for (int c = 0; c < NC; c++) asm volatile("" : "+v"(off[c]));
    }
    // the same unpacking (mins not folded) in pieces 0..8 a caller spreads between other work, and where the compiler is
    // left to place it (Q4_K)
    struct Scales {
        BlockScales s;
        ScalePairs p;
    };
    static __device__ __forceinline__ Scales scales(const Raw &R, int) {
        static_assert(!Q5, "in pieces: Q4_K's planes only");
        const BlockScales s = block_scales(R.wh);
        return {s, scale_pairs(s)};
    }
    static __device__ __forceinline__ void unpack_piece(int i, const Raw &R, const Scales &c, int lg, int, BPlanes &B) {
        static_assert(!Q5, "in pieces: Q4_K's planes only");
        if (i == 0) unpack_pair_free(R.q0, c.p.p0, c.p.p1, B.H0, B.L0, B.H1, B.L1);
        if (i == 2) unpack_pair_free(R.q1, c.p.p2, c.p.p3, B.H2, B.L2, B.H3, B.L3);
        if (i == 4) unpack_pair_free(R.q2, c.p.p4, c.p.p5, B.H4, B.L4, B.H5, B.L5);
        if (i == 6) unpack_pair_free(R.q3, c.p.p6, c.p.p7, B.H6, B.L6, B.H7, B.L7);
        if (i == 8) unpack_rest(R.wh, c.s, lg, B);
    }
};
// Q6_K: 32 rows x 128 bytes of ql (four requests), 64 of qh (two), 16 of scales and the four bytes that hold the block's
// d and its even or odd neighbour's.  A row's pieces of ql and qh are stored XOR-swizzled by the row number, so that 32
// rows' reads of one logical piece fall in different banks while every request still covers whole rows.
template <>
struct WeightSide<FRK_KIND_Q6_K> {
    static constexpr int QH = 32 * 128, SC = QH + 32 * 64, D = SC + 32 * 16;
    static constexpr int SLOT = D + 32 * 4, SHIFT = 8, REQUESTS = 8;
    static constexpr bool MINS = false;
    using Raw = RawBlock6;
    uint32_t ql_off[4], qh_off[2], row_off;
    const uint8_t *ql, *qh, *sc, *d;
    __device__ __forceinline__ void offsets(uint32_t stride, int last_row, int lane) {
        auto row = [&](int r) { return (uint32_t)min(r, last_row) * stride; };
#pragma unroll
        for (int c = 0; c < 4; c++)  // 8 rows a request; piece p of an LDS row is piece p ^ (row & 7)
            ql_off[c] = row(8 * c + (lane >> 3)) + (uint32_t)((lane & 7) ^ (lane >> 3)) * 16 + 4096u - 1024u * c;
#pragma unroll
        for (int c = 0; c < 2; c++) {  // 16 rows a request; piece p is piece p ^ ((row >> 1) & 3)
            const int r = 16 * c + (lane >> 2);
            qh_off[c] = row(r) + (uint32_t)((lane & 3) ^ ((r >> 1) & 3)) * 16 + 4096u - 1024u * c;
        }
        row_off = row(lane & 31);
    }
    template <class Args>
    __device__ __forceinline__ void point_at(const Args &g, const uint8_t *W, int row_base, int kb) {
        const uint8_t *first = W + (size_t)row_base * g.row_stride;
        ql = (const uint8_t *)scalar_pointer(first + (size_t)kb * 128 - 4096);
        qh = (const uint8_t *)scalar_pointer(first + g.off_qh + (size_t)kb * 64 - 4096);
        sc = (const uint8_t *)scalar_pointer(first + g.off_sc + (size_t)kb * 16);
        d = (const uint8_t *)scalar_pointer(first + g.off_d + (size_t)(kb >> 1) * 4);
    }
    __device__ __forceinline__ void fetch(uint32_t slot, int lane) {
        dma16_run<4>(slot, ql, ql_off[0], ql_off[1], ql_off[2], ql_off[3]);
        dma16_run<2>(slot + QH, qh, qh_off[0], qh_off[1], 0, 0);
        if (lane < 32) {
            dma16_run<1>(slot + SC, sc, row_off, 0, 0, 0);
            dma4(slot + D, d, row_off);
        }
    }
    __device__ __forceinline__ void move_on(int kb) {  // from block kb to the next
        ql += 128, qh += 64, sc += 16;
        d += kb & 1 ? 4 : 0;
    }
    static __device__ __forceinline__ void read(Raw &R, uint32_t slot, int r, int lg) {
        const uint32_t a = slot + r * 128, b = slot + QH + r * 64;
        auto ql_piece = [&](int p) { return a + (uint32_t)((p + lg) ^ (r & 7)) * 16; };
        auto qh_piece = [&](int p) { return b + (uint32_t)((p + lg) ^ ((r >> 1) & 3)) * 16; };
        FRK_DS_READ(R.l0a, ql_piece(0), 0);
        FRK_DS_READ(R.l0b, ql_piece(2), 0);
        FRK_DS_READ(R.l1a, ql_piece(4), 0);
        FRK_DS_READ(R.l1b, ql_piece(6), 0);
        FRK_DS_READ(R.h0, qh_piece(0), 0);
        FRK_DS_READ(R.h1, qh_piece(2), 0);
        FRK_DS_READ(R.sc, slot + SC + r * 16, 0);
        asm volatile("ds_read_b32 %0, %1" : "=v"(R.d2) : "v"(slot + D + r * 4));
        wait_raw<0>(R);
    }
    static __device__ __forceinline__ void unpack(const Raw &R, int lg, int kb, BPlanes &B) {
        const Scales c = scales(R, lg);
#pragma unroll
        for (int i = 0; i < 9; i++) unpack_piece(i, R, c, lg, kb, B);
    }
    __device__ __forceinline__ void pin() {
#pragma unroll
        for (int c = 0; c < 4; c++) asm volatile("" : "+v"(ql_off[c]));
        asm volatile("" : "+v"(qh_off[0]), "+v"(qh_off[1]), "+v"(row_off));
    }
    struct Scales {  // of this lane's half of every sub-block: groups 2j + lg, sub-blocks j = 0 and 1 in bytes 0 and 2, ...
        uint32_t s01, s23, s45, s67;
    };
    static __device__ __forceinline__ Scales scales(const Raw &R, int lg) {
        const uint32_t by = 8u * (uint32_t)lg;
        return {(uint32_t)R.sc.x >> by, (uint32_t)R.sc.y >> by, (uint32_t)R.sc.z >> by, (uint32_t)R.sc.w >> by};
    }
    static __device__ __forceinline__ void unpack_piece(int i, const Raw &R, const Scales &c, int, int kb, BPlanes &B) {
        if (i == 0) unpack_sub6<0>(R.l0a, R.h0, c.s01, B.H0, B.L0);
        if (i == 1) unpack_sub6<1>(R.l0b, R.h0, c.s01, B.H1, B.L1);
        if (i == 2) unpack_sub6<2>(R.l0a, R.h0, c.s23, B.H2, B.L2);
        if (i == 3) unpack_sub6<3>(R.l0b, R.h0, c.s23, B.H3, B.L3);
        if (i == 4) unpack_sub6<0>(R.l1a, R.h1, c.s45, B.H4, B.L4);
        if (i == 5) unpack_sub6<1>(R.l1b, R.h1, c.s45, B.H5, B.L5);
        if (i == 6) unpack_sub6<2>(R.l1a, R.h1, c.s67, B.H6, B.L6);
        if (i == 7) unpack_sub6<3>(R.l1b, R.h1, c.s67, B.H7, B.L7);
        if (i == 8) B.d = h2f(kb & 1 ? (uint32_t)R.d2 >> 16 : (uint32_t)R.d2 & 0xffffu);
    }
};

template <int KIND, int RG, int KS, int MT>
struct PipeLds {
    using Side = WeightSide<KIND>;
    static constexpr int NW = RG * KS;
    static constexpr int NT = KS * MT;  // tile slots of a stage
    static constexpr int OFF_BS = NT * 8192;
    static constexpr int A_STAGE = NT * (8192 + (Side::MINS ? 1024 : 0));  // quants [NT][8 slices][1 KB] | sums f16 [NT][1 KB]
    static constexpr int A_STAGES = 3;
    static constexpr int OFF_DA = A_STAGES * A_STAGE;
    static constexpr int DA_STAGE = NT * 128, DA_STAGES = 4;
    static constexpr int OFF_W = OFF_DA + DA_STAGES * DA_STAGE;
    static constexpr size_t BYTES = (size_t)OFF_W + (size_t)NW * Side::SLOT;
    static_assert(BYTES <= 160 * 1024, "LDS of a CU");
};

// A workgroup's entry of the work list.  The last token tile may be split into parts of its own number (k_last: it has fewer rows in
// use, so a part of it may have more blocks): its entries then come behind all others.
struct PipeEntry {
    int part, parts, row_tile, tok_tile;  // part < 0: none
};
template <bool APART>  // whether that may be
__device__ __forceinline__ PipeEntry pipe_entry(const GemmArgs &g) {
    int tok_tiles = g.tok_tiles, i;
    if (!APART || g.k_last == g.k_split) {
        i = deal_entry((int)blockIdx.x, g.row_tiles * tok_tiles * g.k_split);
    } else {
        const int first = g.row_tiles * --tok_tiles * g.k_split;
        i = deal_entry((int)blockIdx.x, first + g.row_tiles * g.k_last);
        if (i >= first) {
            i -= first;
            return {i / g.row_tiles, g.k_last, i % g.row_tiles, tok_tiles};
        }
    }
    if (i < 0) return {-1, 1, 0, 0};
    const int tile = i / tok_tiles, inner = g.parts_inner ? g.k_split : g.row_tiles;
    const int high = tile / inner, low = tile - high * inner;
    return {g.parts_inner ? low : high, g.k_split, g.parts_inner ? high : low, i - tile * tok_tiles};
}

// ACT: the workgroup's token tiles with rows in use (the last one of a batch may have fewer than MT)
template <int KIND, int RG, int KS, int MT, int ACT>
__device__ __forceinline__ void pipe_gemm_tiles(const GemmArgs &g, const PipeEntry &entry) {
    using L = PipeLds<KIND, RG, KS, MT>;
    using Side = typename L::Side;
    constexpr bool MINS = Side::MINS;
    constexpr int FORM = !MINS ? NO_MINS : MT == 4 ? MINS_FOLDED : MINS_APART;
    constexpr int NW = L::NW, NT = L::NT, ROWS = 32 * RG, TM = 32 * MT;
    static_assert(NW == 8 && NT == 4 && (MT == 1 || MT == 2 || MT == 4), "eight wavefronts share the four tile slots of a stage");
    extern __shared__ uint4 smem_gemm[];
    uint8_t *lds = reinterpret_cast<uint8_t *>(smem_gemm);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(lds));
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lg = lane >> 5;
    const int rg = wave % RG, ks = wave / RG;

    // An XCD takes an equal run of the list (part, row tile, token tile), or (row tile, part, token tile): its workgroups share weight rows and, where the
    // blocks are split, the activations of a part or two.  (With XCD x given the row tiles congruent to x mod 8, the busiest
    // one had a round more than the others wherever their number does not divide by eight: 2440 x 12032 in Q5_K at 146
    // tokens, 20 row tiles, 53 -> 33 us; and with the parts in the middle of the list every XCD reads all activations: 1025
    // x 13056 in Q4_K at 105 tokens in eight parts 23.4 -> 21.1.  parts_inner: see pipe_args.)
    const int part = entry.part, row_tile = entry.row_tile, tok0 = entry.tok_tile * TM;
    const int nb = g.nb;
    // this workgroup multiplies blocks kb0 .. kb1 - 1, its KS shares `steps` consecutive ones each (a
    // share that runs out of blocks idles through its last steps)
    const int kb0 = nb * part / entry.parts, kb1 = nb * (part + 1) / entry.parts;
    const int steps = (kb1 - kb0 + KS - 1) / KS;
    const int tile0 = tok0 / 32, last_tile = (g.M - 1) / 32;
    auto tile_of = [&](int slot) { return min(tile0 + slot % MT, last_tile); };  // uniform

    // ---- the fetch side.  Every address is a scalar pointer that moves on by one block a step plus a lane
    // offset that never changes, and a stage of the rings is a scalar offset that rotates: a step's requests
    // cost a handful of scalar instructions.  The first four wavefronts -- the ones the SIMDs' arbiters
    // favour (they are the older of each SIMD's two), which otherwise wait at the step's barrier for the
    // other four -- fetch the activations: wavefront f the record of tile slot f (8 KB of quants, 1 KB of
    // sums), wavefronts 0 and 1 the scales of two slots each.  Every wavefront fetches its own weight rows.
    const bool fetches_acts = wave < NT;
    const bool fetches_scales = wave < (MT == 1 ? 4 : 2);  // (MT 1: two slots are two shares' blocks, not two tiles of one)
    const uint32_t lane16 = (uint32_t)lane * 16;
    const int slot_f = wave & 3, slot_d = MT == 1 ? wave & 3 : (wave & 1) * 2;
    // (a share past its last block keeps requesting that block: nobody multiplies it)
    int next_kb_a = kb0 + (slot_f / MT) * steps;  // the block of this wavefront's activation slot at the next request
    int next_kb_d = kb0 + (slot_d / MT) * steps;
    int next_kb_w = kb0 + ks * steps;
    const uint8_t *src_q = (const uint8_t *)scalar_pointer(reinterpret_cast<const uint8_t *>(g.a.q) +
                                                           ((size_t)tile_of(slot_f) * nb + min(next_kb_a, kb1 - 1)) * 8192);
    const uint8_t *src_s = (const uint8_t *)scalar_pointer(reinterpret_cast<const uint8_t *>(g.a.bs) +
                                                           ((size_t)tile_of(slot_f) * nb + min(next_kb_a, kb1 - 1)) * 1024);
    const uint8_t *src_d = (const uint8_t *)scalar_pointer(reinterpret_cast<const uint8_t *>(g.a.d) +
                                                           ((size_t)tile_of(slot_d) * nb + min(next_kb_d, kb1 - 1)) * 128);
    const uint32_t lane_d = (uint32_t)(lane & 31) * 4 +
                            (MT > 1 && lane >= 32 ? (uint32_t)(tile_of(slot_d + 1) - tile_of(slot_d)) * (uint32_t)nb * 128u : 0u);
    Side wside;
    const int row_base = min(row_tile * ROWS + rg * 32, g.rows - 1);
    wside.offsets((uint32_t)g.row_stride, g.rows - 1 - row_base, lane);
    wside.point_at(g, g.W, row_base, min(next_kb_w, kb1 - 1));
    const uint32_t lds_w = lds0 + L::OFF_W + wave * Side::SLOT;
    // the rings: activations three stages (a step's stage, the next one's, the one being filled), scales four
    uint32_t st_cur = lds0, st_next = lds0 + L::A_STAGE, st_fill = lds0;  // st_fill: where the next request lands
    uint32_t da_fill = lds0 + L::OFF_DA;
    auto fetch_quants = [&](int half) {  // half of the slot's record: 4 KB
        dma16_run<4>(st_fill + slot_f * 8192 + half * 4096, src_q + half * 4096, lane16, lane16, lane16, lane16);
    };
    auto fetch_sums_scales = [&]() {
        if (MINS) dma16_run<1>(st_fill + L::OFF_BS + slot_f * 1024, src_s, lane16, 0, 0, 0);
        if (fetches_scales && (MT > 1 || lane < 32)) dma4(da_fill + slot_d * 128, src_d, lane_d);
    };
    auto acts_fetched = [&]() {  // the request for a step is out: everything moves on to the step after
        const bool adv_a = next_kb_a + 1 < kb1, adv_d = next_kb_d + 1 < kb1;
        next_kb_a++, next_kb_d++;
        src_q += adv_a ? 8192 : 0;
        src_s += adv_a ? 1024 : 0;
        src_d += adv_d ? 128 : 0;
        st_fill = st_fill == lds0 + 2 * L::A_STAGE ? lds0 : st_fill + L::A_STAGE;
        da_fill = da_fill == lds0 + L::OFF_DA + 3 * L::DA_STAGE ? lds0 + L::OFF_DA : da_fill + L::DA_STAGE;
    };
    auto fetch_weights = [&]() {
        wside.fetch(lds_w, lane);
        if (next_kb_w + 1 < kb1) wside.move_on(next_kb_w);
        next_kb_w++;
    };

    v16f sum[ACT];
#pragma unroll
    for (int mt = 0; mt < ACT; mt++) sum[mt] = v16f{0.0f};
    BPlanes B;
    typename Side::Raw R;
    int kb_raw = kb0 + ks * steps;  // the block that leaves the slot next
    // a raw block leaves this wavefront's slot for registers
    auto read_block = [&]() { Side::read(R, lds_w, li, lg); };
    auto unpack = [&]() {
        Side::unpack(R, lg, kb_raw++, B);
        if (FORM == MINS_FOLDED) fold_mins(B);
    };

    // prologue: activations of steps 0 and 1, weights of step 0; then the weights of step 1
    if (fetches_acts) {
        fetch_quants(0), fetch_quants(1), fetch_sums_scales(), acts_fetched();
    }
    fetch_weights();
    if (steps > 1 && fetches_acts) {
        fetch_quants(0), fetch_quants(1), fetch_sums_scales(), acts_fetched();
    }
    // how many requests of a step's activations this wavefront makes (they stay in flight over the step's end)
    const int acts_requests = (fetches_scales ? 9 : fetches_acts ? 8 : 0) + (MINS && fetches_acts ? 1 : 0);
    // where a step's first tile slot of this wavefront's share sits in its stage (lane offsets in)
    const uint32_t rd_q = (uint32_t)(ks * MT) * 8192 + lane16, rd_b = L::OFF_BS + (uint32_t)(ks * MT) * 1024 + lane16;
    const uint32_t rd_d = lds0 + L::OFF_DA + (uint32_t)(ks * MT) * 128 + lg * 16;
    const int my_steps = max(0, min(steps, kb1 - (kb0 + ks * steps)));  // the steps in which this wavefront's share has a block
    TileOperands T;  // the first tile's operands of the step about to run: requested behind the barrier, so that
                     // they travel while the block is unpacked
    wait_vm<0>();
    lds_barrier();
    {
        read_block();
        if (steps > 1) fetch_weights();
        if (my_steps > 0) read_tile<0, MINS>(T, st_cur + rd_q, st_cur + rd_b);
        unpack();
    }

    for (int i = 0; i < steps; i++) {
        const bool active = i < my_steps;
        const uint32_t qa = st_cur + rd_q, ba = st_cur + rd_b;
        const uint32_t sa = rd_d + (uint32_t)(i & 3) * L::DA_STAGE;
        const bool more_acts = i + 2 < steps;
        const bool fetch_now = more_acts && fetches_acts;
        if (active) {
            TileOperands Tn;
            TileTail E;
            // One tile after the other; the second half of a tile's chain requests the next tile's operands
            // into the registers it has read for the last time, and carries the tail of the tile before.
            auto run_tile = [&](auto mt_c) {
                constexpr int mt = decltype(mt_c)::value;
                auto between = [&](int j) {
                    if (mt == 0) {
                        if (fetch_now) {
                            if (j == 1) fetch_quants(0);
                            if (j == 3) fetch_quants(1);
                            if (j == 5) fetch_sums_scales(), acts_fetched();
                        }
                    } else {
                        // the scales of the tile before were the last reads requested ahead of this chain:
                        // they have landed once the chain has waited for everything, in front of MFMA 8, and
                        // only from here on may the compiler touch them
                        if (j == 8) wait_scales<0>(E.S);
                        tail_piece<FORM>(j, E, B, sum[mt > 0 ? mt - 1 : 0]);
                    }
                };
                auto next = [&](int j) {
                    if (mt + 1 < ACT) {
                        constexpr int nx = mt + 1 < ACT ? mt + 1 : mt;
                        if (j == 0) read_tile_operand<nx, 0>(Tn, qa);
                        if (j == 1) read_tile_operand<nx, 1>(Tn, qa);
                        if (j == 2) read_tile_operand<nx, 2>(Tn, qa);
                        if (j == 3) read_tile_operand<nx, 3>(Tn, qa);
                        if (j == 4) read_tile_operand<nx, 4>(Tn, qa);
                        if (j == 5) read_tile_operand<nx, 5>(Tn, qa);
                        if (j == 6) read_tile_operand<nx, 6>(Tn, qa);
                        if (j == 7) read_tile_operand<nx, 7>(Tn, qa);
                    }
                };
                // (a tile after the first finds four more reads behind its own: the scales of the tile before)
                constexpr int LATER = (MINS ? 1 : 0) + (mt > 0 ? 4 : 0);
                E.s1 = tile_chain<LATER, MINS, Side::SHIFT>(T, B, between, next);
                if (MINS) E.bs = T.bs;
                if (MINS && mt + 1 < ACT) {
                    constexpr int nx = mt + 1 < ACT ? mt + 1 : mt;
                    read_tile_sums<nx>(Tn, ba);
                }
                read_tile_scales<mt>(E.S, sa);
                if (mt + 1 < ACT) T = Tn;
            };
            run_tile(std::integral_constant<int, 0>());
            if (ACT > 1) run_tile(std::integral_constant<int, 1 < ACT ? 1 : 0>());
            if (ACT > 2) run_tile(std::integral_constant<int, 2 < ACT ? 2 : 0>());
            if (ACT > 3) run_tile(std::integral_constant<int, 3 < ACT ? 3 : 0>());
            // the last tile's tail is exposed
            wait_scales<0>(E.S);
#pragma unroll
            for (int j = 0; j < 16; j++) tail_piece<FORM>(j, E, B, sum[ACT - 1]);
        } else if (fetch_now) {
            fetch_quants(0), fetch_quants(1), fetch_sums_scales(), acts_fetched();
        }
        if (i + 1 < steps) {
            // step i+1's raw weights (requested a step ago) leave their slot, which is refilled at once;
            // the activations of step i+2, younger than they, may stay in flight
            if (!fetch_now) wait_vm<0>();
            else if (acts_requests == 10) wait_vm<10>();
            else if (acts_requests == 9) wait_vm<9>();
            else wait_vm<8>();
            read_block();
            if (more_acts) fetch_weights();
            lds_barrier();
            st_cur = st_next;
            st_next = st_next == lds0 + 2 * L::A_STAGE ? lds0 : st_next + L::A_STAGE;
            if (i + 1 < my_steps) read_tile<0, MINS>(T, st_cur + rd_q, st_cur + rd_b);
            unpack();
        } else {
            lds_barrier();
        }
    }

    // several shares of the blocks: the later ones' sums go through LDS and are added onto the first's, two and two
    if (KS > 1) {
        float *xch = reinterpret_cast<float *>(lds) + (size_t)rg * (KS - 1) * MT * 16 * 64;
        if (ks > 0) {
#pragma unroll
            for (int mt = 0; mt < ACT; mt++)
#pragma unroll
                for (int r = 0; r < 16; r++) xch[(((ks - 1) * MT + mt) * 16 + r) * 64 + lane] = sum[mt][r];
        }
        __syncthreads();
        if (ks > 0) return;
        static_assert(KS <= 2 || KS == 4, "shares");
#pragma unroll
        for (int mt = 0; mt < ACT; mt++)
#pragma unroll
            for (int r = 0; r < 16; r++) {
                auto share = [&](int k) { return xch[(((k - 1) * MT + mt) * 16 + r) * 64 + lane]; };
                sum[mt][r] += share(1);
                if (KS == 4) sum[mt][r] += share(2) + share(3);
            }
    }
    // store: a lane holds one weight row and 16 tokens per tile
    const int row = row_tile * ROWS + rg * 32 + li;
    float *const dst = entry.parts > 1 ? g.partial + (size_t)part * g.M * g.rows : g.y;
    const int rows_lim = g.rows;
#pragma unroll
    for (int mt = 0; mt < ACT; mt++)
#pragma unroll
        for (int r = 0; r < 16; r++) {
            const int tok = tok0 + mt * 32 + (r >> 2) * 8 + lg * 4 + (r & 3);
            if (row < rows_lim && tok < g.M) dst[(size_t)tok * g.rows + row] = sum[mt][r];
        }
}

template <int KIND, int RG, int KS, int MT>
__device__ __forceinline__ void pipe_gemm(const GemmArgs &g) {
    const PipeEntry entry = pipe_entry<MT == 4>(g);
    if (entry.part < 0) return;  // uniform per workgroup
    const int in_use = (g.M + 31) / 32 - entry.tok_tile * MT;
    if (MT < 4 || in_use >= MT) pipe_gemm_tiles<KIND, RG, KS, MT, MT>(g, entry);
    else if (in_use == 3) pipe_gemm_tiles<KIND, RG, KS, MT, MT == 4 ? 3 : MT>(g, entry);
    else if (in_use == 2) pipe_gemm_tiles<KIND, RG, KS, MT, MT == 4 ? 2 : MT>(g, entry);
    else pipe_gemm_tiles<KIND, RG, KS, MT, MT == 4 ? 1 : MT>(g, entry);
}

// ------------------------------------------------------------------ host side

// The workgroup tile of a batch: 256 rows x 128 tokens, 128 x 64 or 64 x 32, and how many workgroups share a row's
// blocks (their sums, in SPLIT_PARTS_BYTES of memory at most, are added afterwards).
struct PipePlan {
    int rows_wg, tok_wg, k_split, k_last;
};
PipePlan pipe_plan(int kind, size_t rows, size_t M, size_t nb);  // frk_gemm.hip

template <int KIND, int RG, int KS, int MT>
int launch_pipe(void (*kernel)(GemmArgs), const GemmArgs &g, hipStream_t s) {
    constexpr size_t shmem = PipeLds<KIND, RG, KS, MT>::BYTES;
    static bool sized = false;  // a benign race: every thread sets the same attribute
    if (!sized) {
        hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, (int)shmem);
        if (e != hipSuccess) return set_error(FRK_ERR_HIP, "hipFuncSetAttribute(LDS %zu): %s", shmem, hipGetErrorString(e));
        sized = true;
    }
    const unsigned grid = (unsigned)deal_grid(g.row_tiles * ((g.tok_tiles - 1) * g.k_split + g.k_last));
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(512), shmem, s, g);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return set_error(FRK_ERR_HIP, "pipelined GEMM launch: %s", hipGetErrorString(e));
    const size_t n = (size_t)g.M * g.rows, last = (size_t)(g.tok_tiles - 1) * (32 * MT) * g.rows;  // where the last token tile begins
    if (g.k_split == g.k_last) return g.k_split > 1 ? launch_sum_parts(g.partial, g.k_split, n, g.y, s) : FRK_OK;
    if (g.k_split == 1) return launch_sum_parts_apart(g.partial, n, last, n, last, 1, g.k_last, g.y, s);
    return launch_sum_parts_apart(g.partial, n, 0, g.k_last > 1 ? n : last, last, g.k_split, g.k_last, g.y, s);
}

int launch_pipe_q6_k(const GemmArgs &g, int rows_wg, hipStream_t s);  // frk_gemm_q6.hip

// what a launch of one matrix over tiled activations needs, by its plan
inline GemmArgs pipe_args(const frk_weights *w, Q8KTiled acts, size_t M, float *y, float *partial, const PipePlan &p) {
    GemmArgs g;
    g.a = acts;
    g.W = w->dev;
    g.row_stride = w->layout.row_stride;
    g.off_qh = (uint32_t)w->layout.off_a;
    g.off_sc = (uint32_t)w->layout.off_b;
    g.off_d = (uint32_t)w->layout.off_c;
    g.rows = (int)w->rows;
    g.nb = (int)(w->cols / QK_K);
    g.M = (int)M;
    g.y = y;
    g.row_tiles = (int)((w->rows + p.rows_wg - 1) / p.rows_wg);
    g.tok_tiles = (int)((M + p.tok_wg - 1) / p.tok_wg);
    g.k_split = p.k_split;
    g.k_last = p.k_last;
    g.partial = partial;
    // A part of a Q6_K row is four runs that end inside cache lines (scales and d a few bytes each: 13 lines for 9 lines'
    // worth of an eighth of 43 blocks): with few activations its row's parts share an L2 instead (4096x11008 at 13 rows 23.7
    // -> 22.7 us; 9 .. 32 rows of 79 drawn matrices 0.2 % in the mean, 33 .. 128 rows would lose 0.8).
    g.parts_inner = w->kind == FRK_KIND_Q6_K && M <= 32;
    return g;
}

}  // namespace frk
