// Family "gemm_f16": the prefill product  y[M,N] (+)= x[M,K] . W^T  on rows that are plain f16 in memory — what ojh_mm
// decodes a block format into, once per call, ahead of a batch (contract of the batch path: f16 activations, the bits
// of `dequant_to_f16`, f32 accumulation; crates/ojas-cuda/src/kernels/gemm_q.rs:1-56).
//
//   gemm_f16d_{128,256x128,256}(xh, w, y, K, N, accum, M)     128 x 128, 256 x 128, 256 x 256 (tokens x rows) per workgroup
//   gemm_f16d_{128,256x128}_kw(xh, w, y, K, N, accum, M)      the same on eight waves, each step's K halved between fours
//   gemm_f16d_128_sk(xh, w, y, K, N, M, nsplit)               grid.y = nsplit: K slices that add into y with f32 atomics
//   grid [8 * ceil(row tiles / 8) * token tiles, 1 | nsplit, 1] x 256 (_kw: 512), K a multiple of 64
//
// Nothing is left to do per weight here, so both operands go from memory straight into LDS (global_load_lds_dwordx4,
// 64 values of a row = 128 bytes per K step, chunk c of row r in slot c ^ ((r >> 1) & 7) so that a fragment read
// touches every bank once) and the loop is copies, fragment reads and matrix instructions.  Four waves, 2 x 2 over the
// tile; a ring of D K steps in LDS: as deep as the tile leaves room for, since one workgroup per CU has nothing else
// to cover a trip to memory with (128 x 128: four steps of 32 KB).  The barrier of a step sits before its last K
// sub-step, whose fragments are in registers by then: its matrix instructions cover the next step's first fragments
// and the requests for the step that takes over the slot.
// `_kw` (what ojh_mm launches but for a short K, and for few tokens on grids that fill the chip: f16d_eight_waves): one wave a SIMD
// waits out every copy and fragment read that is late, and a
// second wave with a tile of its own finds no room in LDS.  Two waves on the same tile, two of a step's four sub-steps each,
// read no more of LDS and fill each other's gaps; their sums meet once, through LDS.  With the decode pass: Q8_0 4096 x 14336
// at 2048 tokens 254 -> 238 us, at 1024 155 -> 149; IQ4_XS 8192^2 at 384 96 -> 92; Q6_K 6914 x 2816 at 333 34.3 -> 33.0.
// What is left is the copies: alone they take 193 of the 218 us of 4096 x 14336 x 2048 (62 of a CU's 130 B/ns from its L2:
// an L2 miss in the step waits on the cache behind it), reads and matrix instructions 174.  All of a step's fragments a step
// ahead instead of a sub-step ahead: no faster (244 against 236 us); operands in panels of 64 values of K: 0 - 2 % here.
// (256 x 256 has no registers for it.)
// Tile -> workgroup (ojk_spread.h): the token tiles of one row tile stay on one XCD, whose L2 fetches its weights once, and
// every XCD has its share of the tiles however few the row tiles are.
#include "ojk_common.h"
#include "ojk_spread.h"

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef float float16v __attribute__((ext_vector_type(16)));

template <int MI, int NJ, int D, int KW, bool SPLITK, bool ACCUM>
__device__ __forceinline__ void gemm_f16_body(const ushort* __restrict__ xh, const ushort* __restrict__ w, float* __restrict__ y,
                                              uint K, uint N, uint M, uint nsplit, uchar* lds) {
    constexpr uint BM = 64u * MI, BN = 64u * NJ, RB = 128u, STAGE = (BM + BN) * RB;                // RB: bytes of a row per K step
    constexpr int XL = 2 * MI / KW, WL = 2 * NJ / KW, NC = XL + WL, Q = MI * NJ;   // copies per wave and step: activations, weights, all; MFMAs per sub-step
    constexpr uint SUB = 4u / KW;                                          // sub-steps of 16 that a wave takes of a K step
    const uint mt = (M + BM - 1u) / BM, nt_ = (N + BN - 1u) / BN;
    uint tn, tm, slice;
    const uint place = (blockIdx.x >> 3) + (SPLITK ? blockIdx.y * (gridDim.x >> 3) : 0u);
    if (!ojk_spread(blockIdx.x & 7u, place, nt_, mt, SPLITK ? nsplit : 1u, tn, tm, slice)) return;
    const uint n0 = tn * BN, m0 = tm * BM;
    uint s_begin = 0, s_end = K >> 6;
    if (SPLITK) {
        const uint per = (s_end + nsplit - 1u) / nsplit;
        s_begin = min(slice * per, s_end);
        s_end = min(s_begin + per, s_end);
        if (s_begin >= s_end) return;
    }
    const uint steps = s_end - s_begin, last = steps - 1u;
    const uint lane = threadIdx.x & 63u, wave = (uint)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint lds0 = (uint)(size_t)(__attribute__((address_space(3))) uchar*)lds;

    // copy i of wave w brings eight rows: lane -> row lane / 8, slot lane % 8
    uint off[NC];
#pragma unroll
    for (int i = 0; i < NC; i++) {
        const bool isx = i < XL;
        const uint r = (wave * (isx ? XL : WL) + (isx ? i : i - XL)) * 8u + (lane >> 3);
        const uint row = isx ? min(m0 + r, M - 1u) : min(n0 + r, N - 1u);
        off[i] = row * K * 2u + (((lane & 7u) ^ ((r >> 1) & 7u)) << 4);
    }
    const uint xdst = lds0 + wave * XL * 1024u, wdst = lds0 + BM * RB + wave * WL * 1024u;
    const uchar* const xb = (const uchar*)xh + (size_t)s_begin * RB;
    const uchar* const wb = (const uchar*)w + (size_t)s_begin * RB;
    // requests past the last step are clamped onto it: every step issues the same NC copies
#define GF_COPY(I, T, SLOT)                                                                                   \
    lds_dma16_s(((I) < XL ? xb : wb) + (size_t)min((T), last) * RB, off[I],                                   \
              ((I) < XL ? xdst + (I) * 1024u : wdst + ((I) - XL) * 1024u) + (SLOT) * STAGE)

    const uint kw = KW > 1 ? wave >> 2 : 0u, wy = (wave >> 1) & 1u, wx = wave & 1u, fr = lane & 31u, kg = lane >> 5, sw = (fr >> 1) & 7u;
    const uint a_off = (wy * 32u * MI + fr) * RB, b_off = BM * RB + (wx * 32u * NJ + fr) * RB;
    float16v acc[MI][NJ];
#pragma unroll
    for (int i = 0; i < MI; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[i][j][v] = 0.0f;
#define GF_READ(SLOT, S, AF, BF)                                                                             \
    do {                                                                                                      \
        const uchar* s_ = lds + (SLOT) * STAGE + (((2u * (kw * SUB + (S)) + kg) ^ sw) << 4);                \
        _Pragma("unroll") for (int i = 0; i < MI; i++) AF[i] = *(const half8*)(s_ + a_off + i * 32u * RB);       \
        _Pragma("unroll") for (int j = 0; j < NJ; j++) BF[j] = *(const half8*)(s_ + b_off + j * 32u * RB);       \
    } while (0)
#define GF_MMA1(q, AF, BF)                                                                                    \
    acc[(q) / NJ][(q) % NJ] = __builtin_amdgcn_mfma_f32_32x32x16_f16(AF[(q) / NJ], BF[(q) % NJ], acc[(q) / NJ][(q) % NJ], 0, 0, 0)
#define GF_SUB(SLOT, S, AF, BF, AN, BN_)                                                                     \
    do {                                                                                                      \
        GF_READ(SLOT, S, AN, BN_);                                                                            \
        _Pragma("unroll") for (int q = 0; q < Q; q++) GF_MMA1(q, AF, BF);                                     \
        _Pragma("unroll") for (int q = 0; q < Q; q++) {                                                       \
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                                                \
            if (q < (MI + NJ + 1) / 2) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);                     \
        }                                                                                                     \
        __builtin_amdgcn_sched_barrier(0);                                                                    \
    } while (0)
    half8 aA[MI], bA[NJ], aB[MI], bB[NJ];
#pragma unroll
    for (int d = 0; d < D; d++)
#pragma unroll
        for (int c = 0; c < NC; c++) GF_COPY(c, (uint)d, (uint)d);
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"((D - 1) * NC) : "memory");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    GF_READ(0u, 0, aA, bA);
    uint slot = 0;
    for (uint t = 0; t < steps; t++) {
        const uint next = slot + 1u == (uint)D ? 0u : slot + 1u;
        __builtin_amdgcn_sched_barrier(0);
        GF_SUB(slot, 1, aA, bA, aB, bB);
        if (KW == 1) {
            GF_SUB(slot, 2, aB, bB, aA, bA);
            GF_SUB(slot, 3, aA, bA, aB, bB);
        }
        // step t + 1 is whole once every wave's own copies of it are, and slot t is free once every wave has read it
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"((D - 2) * NC) : "memory");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        GF_READ(next, 0, aA, bA);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int q = 0; q < Q; q++) {
            GF_MMA1(q, aB, bB);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = (NC * q) / Q; c < (NC * (q + 1)) / Q; c++) GF_COPY(c, t + (uint)D, slot);
            __builtin_amdgcn_sched_barrier(0);
        }
        slot = next;
    }
    // no copy may still be on its way into LDS that the next workgroup owns
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
#undef GF_COPY
#undef GF_READ
#undef GF_MMA1
#undef GF_SUB
    // The two halves of K meet in LDS: each group of waves leaves the token blocks that the other one stores.
    constexpr int IH = KW > 1 ? MI / 2 : 0, IN = KW > 1 ? MI / 2 : MI;     // (token blocks handed over; stored by a wave)
    const int i0 = KW > 1 && kw ? IH : 0;
    if (KW > 1) {
        float4* const mine = (float4*)lds + (size_t)wave * (IH * NJ * 4) * 64u + lane;
        const float4* const theirs = (const float4*)lds + (size_t)(wave ^ 4u) * (IH * NJ * 4) * 64u + lane;
        __syncthreads();
#pragma unroll
        for (int i = 0; i < IH; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float16v& a = kw ? acc[i][j] : acc[IH + i][j];
                    mine[((i * NJ + j) * 4 + v) * 64] = make_float4(a[4 * v], a[4 * v + 1], a[4 * v + 2], a[4 * v + 3]);
                }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < IH; i++)
#pragma unroll
            for (int j = 0; j < NJ; j++) {
                if (kw) acc[i][j] = acc[IH + i][j];
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const float4 o = theirs[((i * NJ + j) * 4 + v) * 64];
                    acc[i][j][4 * v] += o.x; acc[i][j][4 * v + 1] += o.y; acc[i][j][4 * v + 2] += o.z; acc[i][j][4 * v + 3] += o.w;
                }
            }
    }
    // D register v of block (i, j) holds token row 8 (v / 4) + 4 kg + v % 4, output fr
#pragma unroll
    for (int i = 0; i < IN; i++)
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const uint n = n0 + wx * 32u * NJ + 32u * j + fr;
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const uint m = m0 + wy * 32u * MI + 32u * (i0 + i) + 8u * (v >> 2) + 4u * kg + (v & 3u);
                if (m < M && n < N) {
                    float* o = y + (size_t)m * N + n;
                    if (SPLITK) atomicAdd(o, acc[i][j][v]);
                    else if (ACCUM) *o += acc[i][j][v];
                    else *o = acc[i][j][v];
                }
            }
        }
}

#define GEMM_F16_ENTRY(NAME, MI, NJ, D)                                                                       \
    extern "C" __global__ void __launch_bounds__(256) NAME(                                                   \
        const ushort* xh, const ushort* w, float* y, uint K, uint N, uint accum, uint M) {                    \
        __shared__ __attribute__((aligned(1024))) uchar lds[(D) * 64 * ((MI) + (NJ)) * 128];                 \
        if (accum) gemm_f16_body<MI, NJ, D, 1, false, true>(xh, w, y, K, N, M, 1u, lds);                      \
        else gemm_f16_body<MI, NJ, D, 1, false, false>(xh, w, y, K, N, M, 1u, lds);                           \
    }
#define GEMM_F16K_ENTRY(NAME, MI, NJ, D)                                                                      \
    extern "C" __global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) NAME(        \
        const ushort* xh, const ushort* w, float* y, uint K, uint N, uint accum, uint M) {                    \
        __shared__ __attribute__((aligned(1024))) uchar lds[(D) * 64 * ((MI) + (NJ)) * 128];                 \
        if (accum) gemm_f16_body<MI, NJ, D, 2, false, true>(xh, w, y, K, N, M, 1u, lds);                      \
        else gemm_f16_body<MI, NJ, D, 2, false, false>(xh, w, y, K, N, M, 1u, lds);                           \
    }
GEMM_F16_ENTRY(gemm_f16d_128, 2, 2, 4)
GEMM_F16_ENTRY(gemm_f16d_256x128, 4, 2, 3)
GEMM_F16_ENTRY(gemm_f16d_256, 4, 4, 2)
GEMM_F16K_ENTRY(gemm_f16d_128_kw, 2, 2, 4)
GEMM_F16K_ENTRY(gemm_f16d_256x128_kw, 4, 2, 3)
extern "C" __global__ void __launch_bounds__(256) gemm_f16d_128_sk(
    const ushort* xh, const ushort* w, float* y, uint K, uint N, uint M, uint nsplit) {
    __shared__ __attribute__((aligned(1024))) uchar lds[4 * 64 * 4 * 128];
    gemm_f16_body<2, 2, 4, 1, true, true>(xh, w, y, K, N, M, nsplit, lds);
}
