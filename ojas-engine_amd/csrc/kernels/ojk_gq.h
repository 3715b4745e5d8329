// Q4_K super-blocks against 16 tokens on the int8 matrix cores: the pieces shared by the dense
// entries (family "gemm_q8k") and the grouped MoE entries (family "moe").
#pragma once
#include "ojk_common.h"

typedef int gq_i4 __attribute__((ext_vector_type(4)));
typedef float gq_f4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ long gq_pack(uint lo, uint hi) { return (long)(((unsigned long)hi << 32) | lo); }

// Four codes (a byte each, <= 15) times a factor <= 7 given as a pair of equal 16-bit halves: no byte's product
// (<= 105) carries into its neighbour, so one packed 16-bit multiply scales all four.
typedef ushort gq_u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint gq_mul4(uint codes, gq_u16x2 f) {
    return __builtin_bit_cast(uint, __builtin_bit_cast(gq_u16x2, codes) * f);
}

struct GqW {            // lane (n, kg): its bytes of one super-block of row n
    uint4 hdr;          // d, dmin, the 12 scale bytes
    uint2 q[4];         // codes of positions 8 kg .. 8 kg + 7 of each 64-weight chunk (low | high nibbles)
};
__device__ __forceinline__ GqW gq_load(const uchar* blk, uint kg) {
    GqW r;
    r.hdr = *(const uint4*)blk;
#pragma unroll
    for (int c = 0; c < 4; c++) r.q[c] = *(const uint2*)(blk + 16u + 32u * c + 8u * kg);
    return r;
}

// One super-block of a 16-row tile against one pass of 16 tokens:
//   acc[v] += sx * (d * sum_j sc_j idot_j - dmin * sum_j m_j bsum_j)   for token 4 kg + v, row n.
// xp: the lane's 8 bytes of token n at this super-block (byte 8 kg); pq: token n's split sums
// (eight lo parts, eight hi parts); sx16: the super-block's 16 token scales.
__device__ __forceinline__ void gq_superblock(const GqW& cur, const uchar* xp, const uchar* pq, const float* sx16, uint kg,
                                              float (&acc)[4]) {
    const gq_i4 zero = {0, 0, 0, 0};
    const float d = f16_bits_to_f32(cur.hdr.x & 0xFFFFu), dmin = f16_bits_to_f32(cur.hdr.x >> 16);
    // all eight 6-bit scales and mins at once, a byte each (get_scale_min_k4, crates/ojas-formats/src/gguf.rs:1132-1140):
    // sub-blocks 0-3 are the low six bits of bytes 0-3 / 4-7, sub-blocks 4-7 a nibble of bytes 8-11 under
    // the top two bits of bytes 0-3 / 4-7
    const uint sc_lo = cur.hdr.y & 0x3F3F3F3Fu, mn_lo = cur.hdr.z & 0x3F3F3F3Fu;
    const uint sc_hi = (cur.hdr.w & 0x0F0F0F0Fu) | ((cur.hdr.y >> 2) & 0x30303030u);
    const uint mn_hi = ((cur.hdr.w >> 4) & 0x0F0F0F0Fu) | ((cur.hdr.z >> 2) & 0x30303030u);
    int sc[8];
    long B[8];
#pragma unroll
    for (int c = 0; c < 4; c++) {
        sc[c] = (int)((sc_lo >> (8 * c)) & 0xFFu);
        sc[4 + c] = (int)((sc_hi >> (8 * c)) & 0xFFu);
        B[2 * c] = gq_pack(cur.q[c].x & 0x0F0F0F0Fu, cur.q[c].y & 0x0F0F0F0Fu);
        B[2 * c + 1] = gq_pack((cur.q[c].x >> 4) & 0x0F0F0F0Fu, (cur.q[c].y >> 4) & 0x0F0F0F0Fu);
    }
    const long Bm = kg == 0u ? gq_pack(mn_lo, mn_hi) : 0;       // mins 0..7 in bytes 0..7; only positions 0..7 carry them
    int isum[4] = {0, 0, 0, 0};
#pragma unroll
    for (int jj = 0; jj < 8; jj++) {
        const long A = *(const long*)(xp + 32 * jj);
        const gq_i4 D = __builtin_amdgcn_mfma_i32_16x16x32_i8(A, B[jj], zero, 0, 0, 0);
#pragma unroll
        for (int v = 0; v < 4; v++) isum[v] += __mul24(sc[jj], D[v]);
    }
    // (masked, not branched over: a branch here splits the unrolled code into basic blocks and costs registers)
    const long km_ = kg == 0u ? -1l : 0l;
    const long Alo = *(const long*)pq & km_, Ahi = *(const long*)(pq + 8) & km_;
    const gq_i4 Dlo = __builtin_amdgcn_mfma_i32_16x16x32_i8(Alo, Bm, zero, 0, 0, 0);
    const gq_i4 Dhi = __builtin_amdgcn_mfma_i32_16x16x32_i8(Ahi, Bm, zero, 0, 0, 0);
    const float4 sx = *(const float4*)(sx16 + 4u * kg);
    acc[0] += sx.x * (d * (float)isum[0] - dmin * (float)(64 * Dhi[0] + Dlo[0]));
    acc[1] += sx.y * (d * (float)isum[1] - dmin * (float)(64 * Dhi[1] + Dlo[1]));
    acc[2] += sx.z * (d * (float)isum[2] - dmin * (float)(64 * Dhi[2] + Dlo[2]));
    acc[3] += sx.w * (d * (float)isum[3] - dmin * (float)(64 * Dhi[3] + Dlo[3]));
}

// The two planes of one 16-row tile's super-block, for operands that span two sub-blocks (v_mfma_i32_16x16x64_i8): a
// 6-bit scale is 8 sh + sl with both parts <= 7, so BA = sl * code and BB = sh * code fit int8 and
// sum_j sc_j idot_j = 8 D_B + D_A exactly.  A chunk of 64 weights per register quad: the lane's eight low-nibble codes in
// positions 0 .. 7 of its sixteen, its eight high-nibble codes in 8 .. 15.
__device__ __forceinline__ void gq_planes(const GqW& w, gq_i4 (&BA)[4], gq_i4 (&BB)[4]) {
    const uint sc_lo = w.hdr.y & 0x3F3F3F3Fu;
    const uint sc_hi = (w.hdr.w & 0x0F0F0F0Fu) | ((w.hdr.y >> 2) & 0x30303030u);
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const uint se = 2 * c < 4 ? (sc_lo >> (16 * c)) & 0xFFu : (sc_hi >> (16 * (c - 2))) & 0xFFu;
        const uint so = 2 * c < 4 ? (sc_lo >> (16 * c + 8)) & 0xFFu : (sc_hi >> (16 * (c - 2) + 8)) & 0xFFu;
        const gq_u16x2 el = {(ushort)(se & 7u), (ushort)(se & 7u)}, eh = {(ushort)(se >> 3), (ushort)(se >> 3)};
        const gq_u16x2 ol = {(ushort)(so & 7u), (ushort)(so & 7u)}, oh = {(ushort)(so >> 3), (ushort)(so >> 3)};
        const uint2 qq = w.q[c];
        const uint lx = qq.x & 0x0F0F0F0Fu, ly = qq.y & 0x0F0F0F0Fu;
        const uint hx = (qq.x >> 4) & 0x0F0F0F0Fu, hy = (qq.y >> 4) & 0x0F0F0F0Fu;
        BA[c] = (gq_i4){(int)gq_mul4(lx, el), (int)gq_mul4(ly, el), (int)gq_mul4(hx, ol), (int)gq_mul4(hy, ol)};
        BB[c] = (gq_i4){(int)gq_mul4(lx, eh), (int)gq_mul4(ly, eh), (int)gq_mul4(hx, oh), (int)gq_mul4(hy, oh)};
    }
}
// One pass of 16 tokens against those planes: gq_superblock's sums and its last line, bit for bit.
// xp: 16 bytes of token n per chunk, 64 bytes apart, in the planes' order (low-nibble sub-block's eight, then the
// high-nibble one's); pq: token n's split sums; Bm: the eight mins in positions 0 .. 7 of lanes kg = 0, zeros elsewhere.
__device__ __forceinline__ void gq_planes_pass(const gq_i4 (&BA)[4], const gq_i4 (&BB)[4], long Bm, float d, float dmin,
                                               const uchar* xp, const uchar* pq, const float* sx16, uint kg, float (&acc)[4]) {
    const gq_i4 zero = {0, 0, 0, 0};
    const gq_i4 lh = *(const gq_i4*)pq;
    gq_i4 DA = zero, DB = zero;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const gq_i4 A = *(const gq_i4*)(xp + 64 * c);
        DA = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, BA[c], DA, 0, 0, 0);
        DB = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, BB[c], DB, 0, 0, 0);
    }
    const gq_i4 Dlo = __builtin_amdgcn_mfma_i32_16x16x32_i8(gq_pack((uint)lh[0], (uint)lh[1]), Bm, zero, 0, 0, 0);
    const gq_i4 Dhi = __builtin_amdgcn_mfma_i32_16x16x32_i8(gq_pack((uint)lh[2], (uint)lh[3]), Bm, zero, 0, 0, 0);
    const float4 sx = *(const float4*)(sx16 + 4u * kg);
    const float sxv[4] = {sx.x, sx.y, sx.z, sx.w};
#pragma unroll
    for (int v = 0; v < 4; v++) acc[v] += sxv[v] * (d * (float)(8 * DB[v] + DA[v]) - dmin * (float)(64 * Dhi[v] + Dlo[v]));
}

// Two signed digits of twice a product, four products at a time: ev and od hold p + 128 in their 16-bit halves (products
// 0, 2 and 1, 3), p even.  hi takes their upper bytes and lo their lower bytes with the sign bit flipped, so that
// p = 256 hi + lo with both in int8, exactly.
__device__ __forceinline__ void gq_digits(uint ev, uint od, int& hi, int& lo) {
    hi = (int)__builtin_amdgcn_perm(od, ev, 0x07030501u);
    lo = (int)(__builtin_amdgcn_perm(od, ev, 0x06020400u) ^ 0x80808080u);
}
// four codes (a byte each) times f, plus b
__device__ __forceinline__ void gq_scale4(uint codes, gq_u16x2 f, gq_u16x2 b, int& hi, int& lo) {
    const gq_u16x2 ev = __builtin_bit_cast(gq_u16x2, codes & 0x00FF00FFu) * f + b;
    const gq_u16x2 od = __builtin_bit_cast(gq_u16x2, __builtin_amdgcn_perm(0u, codes, 0x0C030C01u)) * f + b;
    gq_digits(__builtin_bit_cast(uint, ev), __builtin_bit_cast(uint, od), hi, lo);
}
