// Family "moe": router and grouped expert FFN on raw Q4_K expert tensors.
//
// Semantics (reference: router crates/ojas-cuda/src/kernels/moe.rs:45-70; expert FFN
// crates/ojas-cpu/src/cpu_glm.rs:551-582, batched per-assignment GPU form
// crates/ojas-metal/src/kernels/moe.rs:199-272):
//   idx, wgt = top-KSEL of softmax(logits), lowest index wins ties, weights renormalised
//   for every assignment a = (token t, slot j), e = idx[a]:
//       act[a] = silu(Wg_e x_t) * (Wu_e x_t);   dv[a] = Wd_e act[a]
//   y[t] (+)= sum_j wgt[t][j] * dv[t*KSEL + j]           (slot order, f32)
// with every matvec in the CPU reference's arithmetic (activations quantized per 256 by quant_q8k,
// integer dots, crates/ojas-cpu/src/cpu_math.rs:539-635).
//
// The reference launches one workgroup column per assignment and leans on the cache for experts
// shared by several tokens.  Here assignments are grouped by expert first (moe_group: counting
// sort -> per-expert offsets + assignment list), and one launch per projection walks the
// experts: a wave loads its rows of expert e once into registers and runs them against every
// token routed to e, so an expert's bytes cross HBM once however many tokens chose it.
//
//   moe_topk(lg, idx, wgt, E, KSEL)                          one token, 1 x 64 threads
//   moe_topk_m(lg, idx, wgt, E, KSEL)                        grid = tokens
//   moe_group(idx, counts, offsets, list, NA, E)             1 x 256 threads; NA = tokens*KSEL
//   moe_gu_q4k_m(xq, xs, wg, wu, act, offsets, list, K, N, KSEL, NA)   grid (ceil(N/8), E)
//   moe_down_{q4k,q5k}_m(aq, as, wd, dv, offsets, list, K, N, NA)      grid (ceil(N/16), E); ceil(N/32) for K <= 1024
//   moe_combine(dv, wgt, y, T, KSEL, D, ACC)                 grid ceil(T*D/256)
//   moe_topk_quant, moe_gu_q4k_{mi,mil,ti}, moe_down_*_{mi,ti}  the router with the quantizer; products that find their assignments
//   moe_gu_q4k_dec(x, wg, wu, act, idx, K, N, KSEL, NA, E)   grid (ceil(N/8), NA): few tokens, f32 in
//   moe_gu_q4k_decr(x, wg, wu, act, lg, idx, wgt, K, N, KSEL, NA, E)  the same with the router inside (writes idx, wgt)
//   moe_down_{q4k,q5k}_dec(act, wd, idx, wgt, y, K, N, KSEL, E, ACC)  grid (ceil(N/8), T): down + weighted sum
//   moe_gu_q4k_slots(x, arena_g, arena_u, act, off_g, off_u, K, N, KSEL, NA, LIM_G, LIM_U)   the decode form over
//   moe_down_q4k_slots(act, arena, off_d, wgt, y, K, N, KSEL, LIM, ACC)                     streamed experts (u64 byte offsets)
//   moe_gu_q4k_mm / moe_down_q4k_mm, moe_gu_q4k_mt / moe_down_q4k_mt (same arguments as the _m entries)
//                                                            grid (ceil(N/16), E): the int8 matrix-core form
#include "ojk_common.h"
#include "ojk_q4k_dot.h"
#include "ojk_gq.h"
#include "ojk_moe_rows.h"
#include <type_traits>

// ------------------------------------------------------------------ router
// KSEL dependent rounds, each a maximum over the wave, are what the router waits for.  Probabilities are never negative, so
// their bits order like integers: the maxima are integer ones (no canonicalising, the last three steps on the scalar unit),
// and the winner is a vote on equality.  A NaN or infinite logit makes every probability NaN: then nothing is chosen (index
// ~0, weights 1 / KSEL).
template <int NI>
__device__ __forceinline__ void moe_topk_lanes(const float* __restrict__ lg, uint* __restrict__ idx,
                                               float* __restrict__ wgt, uint E, uint KSEL) {
    // one wave per token; lane l owns experts l, l+64, ... (E <= 64 NI)
    const uint lane = threadIdx.x & 63u;
    const int NONE = 0xBF800000;    // -1.0f: taken, or no expert
    float p[NI];
    float mx = -3.4028235e38f;
#pragma unroll
    for (int i = 0; i < NI; i++) {
        uint e = lane + 64u * i;
        p[i] = e < E ? lg[e] : -3.4028235e38f;
        mx = fmaxf(mx, p[i]);
    }
    mx = wave_max(mx);
    float sum = 0.0f;
#pragma unroll
    for (int i = 0; i < NI; i++) {
        uint e = lane + 64u * i;
        p[i] = e < E ? expf(p[i] - mx) : -1.0f;
        if (e < E) sum += p[i];
    }
    sum = wave_sum(sum);
    int key[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const float q = p[i] / sum;
        key[i] = lane + 64u * i < E && q >= 0.0f ? __float_as_int(q) : NONE;
    }
    float wsum = 0.0f, mine = 0.0f;
    uint mine_idx = 0;
    for (uint j = 0; j < KSEL; j++) {
        int best = key[0];
#pragma unroll
        for (int i = 1; i < NI; i++) best = max(best, key[i]);
        const int m2 = wave_max_i32(best);
        // lowest index among the experts holding the maximum: an expert's index is lane + 64 i, so the lowest i with any
        // such lane decides, and within it the lowest lane — one vote per i and scalar bit scans instead of a second
        // reduction across the wave
        uint win = 0xFFFFFFFFu;
#pragma unroll
        for (int i = NI - 1; i >= 0; i--) {
            const unsigned long long vote = __ballot(key[i] == m2);
            if (vote) win = (uint)__builtin_ctzll(vote) + 64u * (uint)i;
        }
        if (m2 < 0) win = 0xFFFFFFFFu;
        wsum += __int_as_float(m2);
        if (lane == j) { mine = __int_as_float(m2); mine_idx = win; }
#pragma unroll
        for (int i = 0; i < NI; i++)
            if (lane + 64u * i == win) key[i] = NONE;
    }
    if (lane < KSEL) {
        idx[lane] = mine_idx;
        wgt[lane] = mine / wsum;
    }
}

__device__ __forceinline__ void moe_topk_body(const float* __restrict__ lg, uint* __restrict__ idx,
                                              float* __restrict__ wgt, uint E, uint KSEL) {
    if (E <= 128u) moe_topk_lanes<2>(lg, idx, wgt, E, KSEL);
    else if (E <= 256u) moe_topk_lanes<4>(lg, idx, wgt, E, KSEL);
    else moe_topk_lanes<16>(lg, idx, wgt, E, KSEL);
}

extern "C" __global__ void __launch_bounds__(64)
moe_topk(const float* lg, uint* idx, float* wgt, uint E, uint KSEL) {
    moe_topk_body(lg, idx, wgt, E, KSEL);
}
extern "C" __global__ void __launch_bounds__(64)
moe_topk_m(const float* lg, uint* idx, float* wgt, uint E, uint KSEL) {
    const size_t t = blockIdx.x;
    moe_topk_body(lg + t * E, idx + t * KSEL, wgt + t * KSEL, E, KSEL);
}

// ---- the reference's other routers (Metal twins crates/ojas-metal/src/kernels/moe.rs:130-150, :531-551) ----
//   moe_topk_nonorm(lg, idx, wgt, E, KSEL)                     DeepSeek-V2: softmax, top-KSEL, the raw probabilities
//   moe_topk_v3(lg, bias, idx, wgt, E, KSEL, RSCALE, NORM)     DeepSeek-V3 / GLM: s = sigmoid(logit); experts chosen by
//       s + bias (strict '>', lowest index wins ties); weight = s of the chosen, times 1 / (their sum) when NORM and the
//       sum is positive, times the routed scaling factor (RSCALE: its f32 bits) — crates/ojas-cpu/src/cpu_glm.rs:526-548
// grid [tokens,1,1] x 64: token t reads lg + t E and writes idx / wgt + t KSEL (one token: grid [1,1,1]).
template <int NI, bool V3>
__device__ __forceinline__ void moe_topk_alt_lanes(const float* __restrict__ lg, const float* __restrict__ bias,
                                                   uint* __restrict__ idx, float* __restrict__ wgt, uint E, uint KSEL,
                                                   float rscale, uint norm) {
    const uint lane = threadIdx.x & 63u;
    float ch[NI], val[NI];      // what the experts are chosen by; what a chosen expert's weight is made of
    float sum = 1.0f;
    if (V3) {
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const uint e = lane + 64u * i;
            const float sg = e < E ? 1.0f / (1.0f + expf(-lg[e])) : 0.0f;
            val[i] = sg;
            ch[i] = e < E ? sg + bias[e] : -3.4028235e38f;
        }
    } else {
        float mx = -1e30f;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const uint e = lane + 64u * i;
            ch[i] = e < E ? lg[e] : -3.4028235e38f;
            if (e < E) mx = fmaxf(mx, ch[i]);
        }
        mx = wave_max(mx);
        sum = 0.0f;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const uint e = lane + 64u * i;
            ch[i] = e < E ? expf(ch[i] - mx) : -3.4028235e38f;
            val[i] = ch[i];
            if (e < E) sum += ch[i];
        }
        sum = wave_sum(sum);
    }
    float wsum = 0.0f, mine = 0.0f;
    uint mine_idx = 0;
    for (uint j = 0; j < KSEL; j++) {
        float bv = V3 ? -1e30f : -1.0f, bval = 0.0f;
        uint bi = 0xFFFFFFFFu;
#pragma unroll
        for (int i = 0; i < NI; i++)
            if (ch[i] > bv) { bv = ch[i]; bval = val[i]; bi = lane + 64u * i; }
        const float m2 = wave_max(bv);
        uint cand = (bv == m2 && bi != 0xFFFFFFFFu) ? bi : 0xFFFFFFFFu;
        cand = min(cand, (uint)dpp_i32<OJK_DPP_QUAD_XOR1>((int)cand));
        cand = min(cand, (uint)dpp_i32<OJK_DPP_QUAD_XOR2>((int)cand));
        cand = min(cand, (uint)dpp_i32<OJK_DPP_ROW_HALF_MIRROR>((int)cand));
        cand = min(cand, (uint)dpp_i32<OJK_DPP_ROW_MIRROR>((int)cand));
        const uint c0 = (uint)__builtin_amdgcn_readlane((int)cand, 0), c1 = (uint)__builtin_amdgcn_readlane((int)cand, 16);
        const uint c2 = (uint)__builtin_amdgcn_readlane((int)cand, 32), c3 = (uint)__builtin_amdgcn_readlane((int)cand, 48);
        const uint win = min(min(c0, c1), min(c2, c3));
        // the winner's value (its lane holds it): all lanes learn it
        const uint wl = win & 63u;
        float wv = 0.0f;
#pragma unroll
        for (int i = 0; i < NI; i++)
            if (lane + 64u * i == win) wv = val[i];
        wv = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wv), (int)__builtin_amdgcn_readfirstlane((int)wl)));
        (void)bval;
        wsum += wv;
        if (lane == j) { mine = wv; mine_idx = win; }
#pragma unroll
        for (int i = 0; i < NI; i++)
            if (lane + 64u * i == win) ch[i] = V3 ? -1e30f : -1.0f;
    }
    if (lane < KSEL) {
        idx[lane] = mine_idx;
        if (V3) {
            const float inv = (norm != 0u && wsum > 0.0f) ? 1.0f / wsum : 1.0f;
            wgt[lane] = mine * inv * rscale;
        } else {
            wgt[lane] = mine / sum;
        }
    }
}

extern "C" __global__ void __launch_bounds__(64)
moe_topk_nonorm(const float* lg, uint* idx, float* wgt, uint E, uint KSEL) {
    const size_t t = blockIdx.x;
    if (E <= 128u) moe_topk_alt_lanes<2, false>(lg + t * E, nullptr, idx + t * KSEL, wgt + t * KSEL, E, KSEL, 1.0f, 0u);
    else if (E <= 256u) moe_topk_alt_lanes<4, false>(lg + t * E, nullptr, idx + t * KSEL, wgt + t * KSEL, E, KSEL, 1.0f, 0u);
    else moe_topk_alt_lanes<16, false>(lg + t * E, nullptr, idx + t * KSEL, wgt + t * KSEL, E, KSEL, 1.0f, 0u);
}
extern "C" __global__ void __launch_bounds__(64)
moe_topk_v3(const float* lg, const float* bias, uint* idx, float* wgt, uint E, uint KSEL, uint RSCALE, uint NORM) {
    const size_t t = blockIdx.x;
    const float rs = __uint_as_float(RSCALE);
    if (E <= 128u) moe_topk_alt_lanes<2, true>(lg + t * E, bias, idx + t * KSEL, wgt + t * KSEL, E, KSEL, rs, NORM);
    else if (E <= 256u) moe_topk_alt_lanes<4, true>(lg + t * E, bias, idx + t * KSEL, wgt + t * KSEL, E, KSEL, rs, NORM);
    else moe_topk_alt_lanes<16, true>(lg + t * E, bias, idx + t * KSEL, wgt + t * KSEL, E, KSEL, rs, NORM);
}

// ------------------------------------------------------------------ grouping
// Counting sort of the NA assignments by expert: counts[E], offsets[E+1], list[NA] (assignment
// ids, expert-major; the order inside an expert's group is arbitrary and has no effect on the
// results, which are stored per assignment).  One workgroup; E <= 1024.  An index past the last expert counts as the last
// one, as in the decode form: the router writes ~0 where it chose nothing, and what is added up behind the products has to be
// this call's.  (Clamped once all are loaded: inside the condition of its load each would be waited for by itself.)
__device__ __forceinline__ void moe_group_body(const uint* __restrict__ idx, uint* __restrict__ counts, uint* __restrict__ offsets,
                                               uint* __restrict__ list, uint NA, uint E, uint* cnt, uint* off) {
    const uint tid = threadIdx.x;
    for (uint e = tid; e < E; e += 256u) cnt[e] = 0u;
    __syncthreads();
    // (eight loads in flight per thread: one at a time, each pass over the assignments cost a round trip to memory per
    // 256 of them — 8 us per pass at 2048)
    for (uint a0 = tid; a0 < NA; a0 += 8u * 256u) {
        uint e[8];
#pragma unroll
        for (int u = 0; u < 8; u++) e[u] = idx[min(a0 + (uint)u * 256u, NA - 1u)];
#pragma unroll
        for (int u = 0; u < 8; u++) e[u] = a0 + (uint)u * 256u < NA ? min(e[u], E - 1u) : 0xFFFFFFFFu;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (e[u] < E) atomicAdd(&cnt[e[u]], 1u);
    }
    __syncthreads();
    {
        // exclusive prefix sums of the counts: a thread takes four consecutive experts (E <= 1024), the threads' totals
        // are scanned across the wave by shuffles and across the four waves through off[1024] .. (free until the end)
        const uint lane = tid & 63u, wv = tid >> 6;
        uint c[4], local = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            c[i] = 4u * tid + (uint)i < E ? cnt[4u * tid + (uint)i] : 0u;
            local += c[i];
        }
        uint incl = local;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const uint up = (uint)__shfl_up((int)incl, d);
            if (lane >= (uint)d) incl += up;
        }
        __shared__ uint wtot[4];
        if (lane == 63u) wtot[wv] = incl;
        __syncthreads();
        uint base = 0;
        for (uint w = 0; w < wv; w++) base += wtot[w];
        uint run = base + incl - local;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            if (4u * tid + (uint)i < E) off[4u * tid + (uint)i] = run;
            run += c[i];
        }
        if (tid == 255u) off[E] = run;      // thread 255 ends at the grand total
    }
    __syncthreads();
    for (uint e = tid; e <= E; e += 256u) {
        offsets[e] = off[e];
        if (e < E) counts[e] = cnt[e];
    }
    for (uint e = tid; e < E; e += 256u) cnt[e] = 0u;  // reused as the per-expert cursor
    __syncthreads();
    for (uint a0 = tid; a0 < NA; a0 += 8u * 256u) {
        uint e[8];
#pragma unroll
        for (int u = 0; u < 8; u++) e[u] = idx[min(a0 + (uint)u * 256u, NA - 1u)];
#pragma unroll
        for (int u = 0; u < 8; u++) e[u] = a0 + (uint)u * 256u < NA ? min(e[u], E - 1u) : 0xFFFFFFFFu;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (e[u] < E) list[off[e[u]] + atomicAdd(&cnt[e[u]], 1u)] = a0 + (uint)u * 256u;
    }
}
extern "C" __global__ void __launch_bounds__(256)
moe_group(const uint* __restrict__ idx, uint* __restrict__ counts, uint* __restrict__ offsets,
          uint* __restrict__ list, uint NA, uint E) {
    __shared__ uint cnt[1024];
    __shared__ uint off[1025];
    moe_group_body(idx, counts, offsets, list, NA, E, cnt, off);
}

// ------------------------------------------------------------------ grouped gate / up
// Block (rb, e): 4 waves x 2 rows = 8 rows of expert e's gate and up.  K must be a multiple of
// 256; a wave walks K in steps of 8 super-blocks (one step for the usual hidden sizes).
extern "C" __global__ void __launch_bounds__(256)
moe_gu_q4k_m(const signed char* __restrict__ xq, const float* __restrict__ xs, const uchar* __restrict__ wg,
             const uchar* __restrict__ wu, float* __restrict__ act, const uint* __restrict__ offsets,
             const uint* __restrict__ list, uint K, uint N, uint KSEL, uint NA) {
    const uint e = blockIdx.y;
    const uint a0 = min(offsets[e], NA), a1 = min(offsets[e + 1], NA);
    if (a0 >= a1) return;
    const uint lane = threadIdx.x & 63u;
    const uint row0 = (blockIdx.x * 4u + (threadIdx.x >> 6)) * 2u;
    if (row0 >= N) return;
    const uint nsb = K >> 8, g = lane >> 3, l = lane & 7u, c = l >> 1;
    const size_t rb = (size_t)nsb * Q4K_BYTES;
    const uchar* g0 = wg + ((size_t)e * N + row0) * rb;
    const uchar* u0 = wu + ((size_t)e * N + row0) * rb;
    const bool two = row0 + 1u < N;
    const size_t r1 = two ? rb : 0;
    if (nsb <= 8u) {
        // the whole row fits one step: weights stay in registers across the expert's tokens
        const bool on = g < nsb;
        const size_t o = (size_t)(on ? g : 0u) * Q4K_BYTES;
        uint4 hg0 = *(const uint4*)(g0 + o), qg0 = *(const uint4*)(g0 + o + 16u + l * 16u);
        uint4 hg1 = *(const uint4*)(g0 + r1 + o), qg1 = *(const uint4*)(g0 + r1 + o + 16u + l * 16u);
        uint4 hu0 = *(const uint4*)(u0 + o), qu0 = *(const uint4*)(u0 + o + 16u + l * 16u);
        uint4 hu1 = *(const uint4*)(u0 + r1 + o), qu1 = *(const uint4*)(u0 + r1 + o + 16u + l * 16u);
        for (uint i = a0; i < a1; i++) {
            const uint a = min(list[i], NA - 1u), t = a / KSEL;
            Q4kFrag f = q4k_load_frag(xq + (size_t)t * nsb * 256u, xs + (size_t)t * nsb, on ? g : 0u, l);
            // (lanes past the row's last super-block multiply by a zero scale: a product of zero, and no branch around
            // each of the four dots)
            f.sx = on ? f.sx : 0.0f;
            float vg0 = q4k_lane_dot(hg0, qg0, c, f), vg1 = q4k_lane_dot(hg1, qg1, c, f);
            float vu0 = q4k_lane_dot(hu0, qu0, c, f), vu1 = q4k_lane_dot(hu1, qu1, c, f);
            // the four sums in one pass: lanes 0 / 1 end with the gate sums of the two rows, lanes 2 / 3 with the up sums
            const float tot = wave_sum4(vg0, vg1, vu0, vu1, lane);
            const float upv = dpp_f32<OJK_DPP_QUAD_XOR2>(tot);
            if (lane < (two ? 2u : 1u)) act[(size_t)a * N + row0 + lane] = (tot / (1.0f + expf(-tot))) * upv;
        }
    } else {
        for (uint i = a0; i < a1; i++) {
            const uint a = min(list[i], NA - 1u), t = a / KSEL;
            float vg0 = 0.0f, vg1 = 0.0f, vu0 = 0.0f, vu1 = 0.0f;
            for (uint sb = g; sb < nsb; sb += 8u) {
                const size_t o = (size_t)sb * Q4K_BYTES;
                Q4kFrag f = q4k_load_frag(xq + (size_t)t * nsb * 256u, xs + (size_t)t * nsb, sb, l);
                vg0 += q4k_lane_dot(*(const uint4*)(g0 + o), *(const uint4*)(g0 + o + 16u + l * 16u), c, f);
                vg1 += q4k_lane_dot(*(const uint4*)(g0 + r1 + o), *(const uint4*)(g0 + r1 + o + 16u + l * 16u), c, f);
                vu0 += q4k_lane_dot(*(const uint4*)(u0 + o), *(const uint4*)(u0 + o + 16u + l * 16u), c, f);
                vu1 += q4k_lane_dot(*(const uint4*)(u0 + r1 + o), *(const uint4*)(u0 + r1 + o + 16u + l * 16u), c, f);
            }
            const float tot = wave_sum4(vg0, vg1, vu0, vu1, lane);
            const float upv = dpp_f32<OJK_DPP_QUAD_XOR2>(tot);
            if (lane < (two ? 2u : 1u)) act[(size_t)a * N + row0 + lane] = (tot / (1.0f + expf(-tot))) * upv;
        }
    }
}

// ------------------------------------------------------------------ grouped down
// Block (rb, e): 4 waves x 4 rows = 16 rows of expert e's down projection, against the quantized
// act of every assignment routed to e.  dv[a][n] holds the unweighted result.
template <class W>
__device__ __forceinline__ void moe_down_m_body(const signed char* __restrict__ aq, const float* __restrict__ as_,
                                                const uchar* __restrict__ wd, float* __restrict__ dv,
                                                const uint* __restrict__ offsets, const uint* __restrict__ list,
                                                uint K, uint N, uint NA) {
    const uint e = blockIdx.y;
    const uint a0 = min(offsets[e], NA), a1 = min(offsets[e + 1], NA);
    if (a0 >= a1) return;
    const uint lane = threadIdx.x & 63u;
    const uint nsb = K >> 8, g = lane >> 3, l = lane & 7u, c = l >> 1;
    const size_t rb = (size_t)nsb * W::BYTES;
    if (nsb <= 4u) {
        // A short row (an expert's down projection: 768 = 3 super-blocks) leaves most of a wave idle in
        // the layout below.  Here the wave's halves take different rows: 8 rows per wave, 32 per
        // workgroup, and a half's two 16-lane sums are added as wave_sum adds them.
        const uint hf = lane >> 5, G = g & 3u;
        const uint rowh = (blockIdx.x * 4u + (threadIdx.x >> 6)) * 8u + hf * 4u;     // this half's first row
        const bool on = G < nsb;
        const uchar* wh = wd + ((size_t)e * N + min(rowh, N - 1u)) * rb + (size_t)(on ? G : 0u) * W::BYTES;
        W wr[4];
#pragma unroll
        for (int r = 0; r < 4; r++) wr[r].load(wh + (size_t)min((uint)r, N - 1u - min(rowh, N - 1u)) * rb, l);
        for (uint i = a0; i < a1; i++) {
            const uint a = min(list[i], NA - 1u);
            Q4kFrag f = q4k_load_frag(aq + (size_t)a * nsb * 256u, as_ + (size_t)a * nsb, on ? G : 0u, l);
            f.sx = on ? f.sx : 0.0f;        // lanes without a super-block of the row: products of zero, no branches
            // the half's four rows in one pass: lane j of each row of 16 gets row j's 16-lane sum, the half's two
            // such sums are added as wave_sum adds them
            float v = row16_sum4(wr[0].dot(c, f), wr[1].dot(c, f), wr[2].dot(c, f), wr[3].dot(c, f), lane);
            v += __shfl_xor(v, 16);
            if ((lane & 31u) < 4u && rowh + (lane & 3u) < N) dv[(size_t)a * N + rowh + (lane & 3u)] = v;
        }
        return;
    }
    const uint row0 = (blockIdx.x * 4u + (threadIdx.x >> 6)) * 4u;
    if (row0 >= N) return;
    const uchar* w0 = wd + ((size_t)e * N + row0) * rb;
    if (nsb <= 8u) {
        const bool on = g < nsb;
        const size_t o = (size_t)(on ? g : 0u) * W::BYTES;
        W wr[4];
#pragma unroll
        for (int r = 0; r < 4; r++) wr[r].load(w0 + (size_t)min((uint)r, N - 1u - row0) * rb + o, l);
        for (uint i = a0; i < a1; i++) {
            const uint a = min(list[i], NA - 1u);
            Q4kFrag f = q4k_load_frag(aq + (size_t)a * nsb * 256u, as_ + (size_t)a * nsb, on ? g : 0u, l);
            f.sx = on ? f.sx : 0.0f;
            const float v = wave_sum4(wr[0].dot(c, f), wr[1].dot(c, f), wr[2].dot(c, f), wr[3].dot(c, f), lane);
            if (lane < 4u && row0 + lane < N) dv[(size_t)a * N + row0 + lane] = v;
        }
    } else {
        for (uint i = a0; i < a1; i++) {
            const uint a = min(list[i], NA - 1u);
            float v[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            for (uint sb = g; sb < nsb; sb += 8u) {
                Q4kFrag f = q4k_load_frag(aq + (size_t)a * nsb * 256u, as_ + (size_t)a * nsb, sb, l);
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    W wr;
                    wr.load(w0 + (size_t)min((uint)r, N - 1u - row0) * rb + (size_t)sb * W::BYTES, l);
                    v[r] += wr.dot(c, f);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; r++) {
                float s = wave_sum(v[r]);
                if (lane == 0 && row0 + r < N) dv[(size_t)a * N + row0 + r] = s;
            }
        }
    }
}
extern "C" __global__ void __launch_bounds__(256)
moe_down_q4k_m(const signed char* aq, const float* as_, const uchar* wd, float* dv, const uint* offsets,
               const uint* list, uint K, uint N, uint NA) {
    moe_down_m_body<W4k>(aq, as_, wd, dv, offsets, list, K, N, NA);
}
// the same over Q5_K rows (an expert's down tensor is often kept a step finer than gate / up)
extern "C" __global__ void __launch_bounds__(256)
moe_down_q5k_m(const signed char* aq, const float* as_, const uchar* wd, float* dv, const uint* offsets,
               const uint* list, uint K, uint N, uint NA) {
    moe_down_m_body<W5k>(aq, as_, wd, dv, offsets, list, K, N, NA);
}
// ... and over Q6_K rows (two steps finer)
extern "C" __global__ void __launch_bounds__(256)
moe_down_q6k_m(const signed char* aq, const float* as_, const uchar* wd, float* dv, const uint* offsets,
               const uint* list, uint K, uint N, uint NA) {
    moe_down_m_body<W6k>(aq, as_, wd, dv, offsets, list, K, N, NA);
}

// ------------------------------------------------------------------ decode: a few tokens, two launches
// With one or a few tokens almost every assignment has its expert to itself, so grouping buys
// nothing and the six launches of the grouped pipeline cost more than the bytes.  Here a workgroup
// is addressed by assignment (gate/up) or by token (down), quantizes the activations it needs into
// LDS itself, and the down projection owns all KSEL slots of its rows, so the router-weighted sum
// happens in the same launch, in slot order.  The arithmetic is that of the grouped integer-dot
// kernels step for step: results are bit-identical.
#define MOE_DEC_GU_K 8192u      // longest row of gate/up the decode form stages (bytes of int8 in LDS)
#define MOE_DEC_DOWN_ACT 32768u // most KSEL * K int8 activations the down launch stages

// All 256 threads: quantize n (a multiple of 256) f32 values into q (int8) and s (one scale per
// 256 values) with quant_q8k's rule (crates/ojas-cpu/src/cpu_math.rs:539-563), the operations of
// the quantize_q8k kernel.  A thread owns 8 consecutive values, 32 lanes side by side a segment.
__device__ __forceinline__ uint2 oct_quant_q8k(float4 a, float4 b, float& scale) {
    // (not negative and no NaN, so integer maxima; a segment is a half of the wave, the other may be idle)
    int mi = __float_as_int(fmaxf(fmaxf(amax4(a), amax4(b)), 0.0f));
    mi = max(mi, dpp_i32<OJK_DPP_QUAD_XOR1>(mi));
    mi = max(mi, dpp_i32<OJK_DPP_QUAD_XOR2>(mi));
    mi = max(mi, dpp_i32<OJK_DPP_ROW_HALF_MIRROR>(mi));
    mi = max(mi, dpp_i32<OJK_DPP_ROW_MIRROR>(mi));
    const int first = max(__builtin_amdgcn_readlane(mi, 0), __builtin_amdgcn_readlane(mi, 16));
    const int second = max(__builtin_amdgcn_readlane(mi, 32), __builtin_amdgcn_readlane(mi, 48));
    const float m = __int_as_float((threadIdx.x & 32u) ? second : first);
    scale = m > 0.0f ? __fdiv_rn(m, 127.0f) : 1.0f;
    const float inv = __fdiv_rn(1.0f, scale);
    return make_uint2(q8k_pack4(a, inv), q8k_pack4(b, inv));
}
// (or threads `first` .. of them: a multiple of 32, as is their number `nt`)  DEPTH: trips whose loads are asked for at once
template <int DEPTH = 1>
__device__ __forceinline__ void block_quant_q8k(const float* __restrict__ x, uint n, signed char* q, float* s, uint first = 0u, uint nt = 256u) {
    for (uint base = (threadIdx.x - first) * 8u; base < n; base += 8u * nt * DEPTH) {
        float4 a[DEPTH], b[DEPTH];
#pragma unroll
        for (int i = 0; i < DEPTH; i++) {
            const uint at = min(base + 8u * nt * i, n - 8u);
            a[i] = *(const float4*)(x + at);
            b[i] = *(const float4*)(x + at + 4u);
        }
#pragma unroll
        for (int i = 0; i < DEPTH; i++) {
            const uint at = base + 8u * nt * i;
            if (at >= n) break;
            float scale;
            const uint2 c = oct_quant_q8k(a[i], b[i], scale);
            *(uint2*)(q + at) = c;
            if ((threadIdx.x & 31u) == 0) s[at >> 8] = scale;
        }
    }
}

// Where an assignment's expert starts, in bytes from the tensor (or arena) base.  Resident experts
// are indexed (idx[a] * N rows); streamed experts sit wherever the host's cache put them and come
// as one byte offset per assignment (the reference's `_slots` kernels,
// crates/ojas-cuda/src/kernels/moe.rs:133-174).  Offsets are rounded down to 16 bytes and clamped
// to `lim256` * 256, the last offset at which a whole expert still fits.
__device__ __forceinline__ size_t expert_base(const void* sel, uint a, bool slots, uint e_or_lim, size_t expert_bytes) {
    if (slots) {
        const size_t o = (size_t)((const unsigned long*)sel)[a] & ~(size_t)15;
        return min(o, (size_t)e_or_lim * 256u);
    }
    return (size_t)min(((const uint*)sel)[a], e_or_lim - 1u) * expert_bytes;
}

// Block (rb, a): 4 waves x 2 rows of gate and up of assignment a's expert against token a / KSEL.
// ROUTE: the workgroup routes its token itself first — wave 0 runs the router over lg[t] while the others quantize the
// token, the slot's expert is read from LDS, and one workgroup per token writes idx / wgt out for the down launch (sel_g /
// sel_u are not read).  A serial chain of trips to memory bounds the launch, not its bytes: the logits, the router's rounds, the
// weights they name (128 experts of 2048 x 768, top 8, one token, traced: 9.0 -> 7.0 us with the token quantized beside the
// router, the rounds on integers and a row's next step asked for before the present one is multiplied).
template <bool SLOTS, bool ROUTE = false>
__device__ __forceinline__ void moe_gu_dec_body(const float* __restrict__ x, const uchar* __restrict__ wg,
                                                const uchar* __restrict__ wu, float* __restrict__ act,
                                                const void* __restrict__ sel_g, const void* __restrict__ sel_u,
                                                uint K, uint N, uint KSEL, uint EG, uint EU,
                                                const float* __restrict__ lg = nullptr, uint* __restrict__ idx_out = nullptr,
                                                float* __restrict__ wgt_out = nullptr) {
    __shared__ __align__(16) signed char xq[MOE_DEC_GU_K];
    __shared__ float xs[MOE_DEC_GU_K / 256u];
    __shared__ uint r_idx[64];
    __shared__ float r_wgt[64];
    uint a = blockIdx.y;
    const uint t = a / KSEL;
    if (ROUTE) {
        if (threadIdx.x < 64u) moe_topk_body(lg + (size_t)t * EG, r_idx, r_wgt, EG, KSEL);
        else block_quant_q8k<2>(x + (size_t)t * K, K, xq, xs, 64u, 192u);
        __syncthreads();
        sel_g = sel_u = r_idx;
        a -= t * KSEL;              // the slot: index into the token's own table
    }
    const uint lane = threadIdx.x & 63u;
    const uint row0 = min((blockIdx.x * 4u + (threadIdx.x >> 6)) * 2u, N - 1u);   // surplus waves repeat the last row
    const uint nsb = K >> 8, g = lane >> 3, l = lane & 7u, c = l >> 1;
    const size_t rb = (size_t)nsb * Q4K_BYTES;
    const uchar* g0 = wg + expert_base(sel_g, a, SLOTS, EG, (size_t)N * rb) + (size_t)row0 * rb;
    const uchar* u0 = wu + expert_base(sel_u, a, SLOTS, EU, (size_t)N * rb) + (size_t)row0 * rb;
    const bool two = row0 + 1u < N;
    const size_t r1 = two ? rb : 0;
    W4k wg0, wg1, wu0, wu1;
    const size_t o0 = (size_t)min(g, nsb - 1u) * Q4K_BYTES;
    wg0.load(g0 + o0, l); wg1.load(g0 + r1 + o0, l);
    wu0.load(u0 + o0, l); wu1.load(u0 + r1 + o0, l);
    if (ROUTE) {
        if (blockIdx.x == 0u && a == 0u && threadIdx.x < KSEL) {
            idx_out[(size_t)t * KSEL + threadIdx.x] = r_idx[threadIdx.x];
            wgt_out[(size_t)t * KSEL + threadIdx.x] = r_wgt[threadIdx.x];
        }
    } else {   // the first step's weights are on their way while the activations are quantized
        block_quant_q8k(x + (size_t)t * K, K, xq, xs);
        __syncthreads();
    }
    float vg0 = 0.0f, vg1 = 0.0f, vu0 = 0.0f, vu1 = 0.0f;
    for (uint s0 = 0; s0 < nsb; s0 += 8u) {
        const uint sb = s0 + g;
        W4k ng0 = wg0, ng1 = wg1, nu0 = wu0, nu1 = wu1;
        if (s0 + 8u < nsb) {
            const size_t o = (size_t)min(sb + 8u, nsb - 1u) * Q4K_BYTES;
            ng0.load(g0 + o, l); ng1.load(g0 + r1 + o, l);
            nu0.load(u0 + o, l); nu1.load(u0 + r1 + o, l);
        }
        if (sb < nsb) {
            const Q4kFrag f = q4k_load_frag(xq, xs, sb, l);
            vg0 += wg0.dot(c, f);
            vg1 += wg1.dot(c, f);
            vu0 += wu0.dot(c, f);
            vu1 += wu1.dot(c, f);
        }
        wg0 = ng0; wg1 = ng1; wu0 = nu0; wu1 = nu1;
    }
    // lanes 0 / 1 end with the gate sums of the two rows, lanes 2 / 3 with the up sums
    const float tot = wave_sum4(vg0, vg1, vu0, vu1, lane);
    const float upv = dpp_f32<OJK_DPP_QUAD_XOR2>(tot);
    if (lane < (two ? 2u : 1u)) act[(size_t)blockIdx.y * N + row0 + lane] = (tot / (1.0f + expf(-tot))) * upv;
}
extern "C" __global__ void __launch_bounds__(256)
moe_gu_q4k_dec(const float* x, const uchar* wg, const uchar* wu, float* act, const uint* idx, uint K, uint N, uint KSEL,
               uint NA, uint E) {
    moe_gu_dec_body<false>(x, wg, wu, act, idx, idx, K, N, KSEL, E, E);
}
// The decode form with the router inside: moe_gu_q4k_decr(x, wg, wu, act, lg, idx, wgt, K, N, KSEL, NA, E) — lg: the
// router logits [tokens][E]; idx / wgt [tokens][KSEL] are written (softmax, top KSEL, renormalised: moe_topk's
// arithmetic, the same bits) for the down launch that follows.  One launch less per layer and token.
extern "C" __global__ void __launch_bounds__(256)
moe_gu_q4k_decr(const float* x, const uchar* wg, const uchar* wu, float* act, const float* lg, uint* idx, float* wgt,
                uint K, uint N, uint KSEL, uint NA, uint E) {
    moe_gu_dec_body<false, true>(x, wg, wu, act, nullptr, nullptr, K, N, KSEL, E, E, lg, idx, wgt);
}
extern "C" __global__ void __launch_bounds__(256)
moe_gu_q4k_slots(const float* x, const uchar* arena_g, const uchar* arena_u, float* act, const unsigned long* off_g,
                 const unsigned long* off_u, uint K, uint N, uint KSEL, uint NA, uint LIM_G, uint LIM_U) {
    moe_gu_dec_body<true>(x, arena_g, arena_u, act, off_g, off_u, K, N, KSEL, LIM_G, LIM_U);
}

// Block (rb, t): 8 rows of the down projection for every slot of token t, 2 rows per wave.  The
// workgroup quantizes the token's KSEL act vectors into LDS.  An expert's row is short (K / 256 <= 8
// super-blocks, three at the usual 768), so a wave's eight lane groups take (slot, super-block)
// pairs side by side instead of one slot at a time: group sums go through LDS, lane j rebuilds
// slot j's dot with the association of wave_sum, and the slots are added in order,
//     y[t][row] (=, +=) sum_j wgt[t][j] * (Wd_{idx[t][j]} act[t][j])[row].
// One wave a SIMD and a few KB a wave: trips to memory one behind the other bound it, so everything that the launch reads
// is asked for at its start (the activations four trips at a time, three passes of weights, the slots' weights): the same
// layer 6.8 -> 5.8 us traced.  A wait for the experts' offsets behind the weights' loads, on one wave, had cost all of that.
template <class W, bool SLOTS>
__device__ __forceinline__ void moe_down_dec_body(const float* __restrict__ act, const uchar* __restrict__ wd,
                                                  const void* __restrict__ sel, const float* __restrict__ wgt,
                                                  float* __restrict__ y, uint K, uint N, uint KSEL, uint E, uint ACC) {
    __shared__ __align__(16) signed char aq[MOE_DEC_DOWN_ACT];
    __shared__ float as_[MOE_DEC_DOWN_ACT / 256u];
    __shared__ size_t s_base[64];
    __shared__ __align__(16) float part[4][2][64][8];   // [wave][row][slot][super-block] group sums
    constexpr uint D = 3u, AD = 4u;
    const uint t = blockIdx.y, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint row0 = min(blockIdx.x * 8u + wave * 2u, N - 1u);   // surplus waves repeat the last row
    const bool two = row0 + 1u < N;
    const uint nsb = K >> 8, G = lane >> 3, l = lane & 7u, c = l >> 1;
    const size_t rb = (size_t)nsb * W::BYTES, r1 = two ? rb : 0;
    const uint U = KSEL * nsb;
    // the pair a lane group takes in each pass: eight further on than in the one before (past the last: the last)
    const uint step_j = 8u / nsb, step_s = 8u - step_j * nsb;
    uint un = G, jn = G / nsb, sn = G - jn * nsb;
    const auto advance = [&]() {
        un += 8u; jn += step_j; sn += step_s;
        if (sn >= nsb) { sn -= nsb; jn++; }
    };
    uint j[D], sb[D];
    size_t eb[D];
#pragma unroll
    for (uint i = 0; i < D; i++) {
        j[i] = un < U ? jn : KSEL - 1u;
        sb[i] = un < U ? sn : nsb - 1u;
        eb[i] = expert_base(sel, t * KSEL + j[i], SLOTS, E, (size_t)N * rb);
        advance();
    }
    const size_t eb_lane = expert_base(sel, t * KSEL + min(threadIdx.x, KSEL - 1u), SLOTS, E, (size_t)N * rb);
    const float wl = wgt[(size_t)t * KSEL + min(lane, KSEL - 1u)];
    float acc0 = 0.0f, acc1 = 0.0f;
    if (ACC) {
        acc0 = y[(size_t)t * N + row0];
        acc1 = y[(size_t)t * N + row0 + (two ? 1u : 0u)];
    }
    const float* at = act + (size_t)t * KSEL * K;
    float4 xa[AD], xb[AD];
#pragma unroll
    for (uint i = 0; i < AD; i++) {
        const uint p = min(threadIdx.x * 8u + 2048u * i, KSEL * K - 8u);
        xa[i] = *(const float4*)(at + p);
        xb[i] = *(const float4*)(at + p + 4u);
    }
    if (threadIdx.x < KSEL) s_base[threadIdx.x] = eb_lane;
    W w0[D], w1[D];
    const uchar* const wrow = wd + (size_t)row0 * rb;
#pragma unroll
    for (uint i = 0; i < D; i++) {
        const uchar* w = wrow + eb[i] + (size_t)sb[i] * W::BYTES;
        w0[i].load(w, l);
        w1[i].load(w + r1, l);
    }
#pragma unroll
    for (uint i = 0; i < AD; i++) {
        const uint p = threadIdx.x * 8u + 2048u * i;
        if (p < KSEL * K) {
            float scale;
            const uint2 q = oct_quant_q8k(xa[i], xb[i], scale);
            *(uint2*)(aq + p) = q;
            if ((threadIdx.x & 31u) == 0) as_[p >> 8] = scale;
        }
    }
    if (KSEL * K > 2048u * AD)
        block_quant_q8k(at + 2048u * AD, KSEL * K - 2048u * AD, aq + 2048u * AD, as_ + 8u * AD);
    __syncthreads();
    for (uint u0 = 0; u0 < U; u0 += 8u * D) {
#pragma unroll
        for (uint i = 0; i < D; i++) {
            const uint ui = u0 + 8u * i;
            if (ui >= U) break;
            const Q4kFrag f = q4k_load_frag(aq + (size_t)j[i] * K, as_ + (size_t)j[i] * nsb, sb[i], l);
            const float v0 = oct_sum(w0[i].dot(c, f)), v1 = oct_sum(w1[i].dot(c, f));
            if (ui + G < U && l == 0) {
                part[wave][0][j[i]][sb[i]] = v0;
                part[wave][1][j[i]][sb[i]] = v1;
            }
            if (ui + 8u * D < U) {
                j[i] = un < U ? jn : KSEL - 1u;
                sb[i] = un < U ? sn : nsb - 1u;
                const uchar* w = wrow + s_base[j[i]] + (size_t)sb[i] * W::BYTES;
                w0[i].load(w, l);
                w1[i].load(w + r1, l);
                advance();
            }
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // lane j: slot j's two dots, summed like wave_sum sums the eight groups of a wave
    float d0 = 0.0f, d1 = 0.0f;
    if (lane < KSEL) {
        float4 p[4];
        p[0] = *(const float4*)&part[wave][0][lane][0]; p[1] = *(const float4*)&part[wave][0][lane][4];
        p[2] = *(const float4*)&part[wave][1][lane][0]; p[3] = *(const float4*)&part[wave][1][lane][4];
        float s0[8] = {p[0].x, p[0].y, p[0].z, p[0].w, p[1].x, p[1].y, p[1].z, p[1].w};
        float s1[8] = {p[2].x, p[2].y, p[2].z, p[2].w, p[3].x, p[3].y, p[3].z, p[3].w};
#pragma unroll
        for (uint k = 1; k < 8; k++) {      // past the row: never written
            s0[k] = k < nsb ? s0[k] : 0.0f;
            s1[k] = k < nsb ? s1[k] : 0.0f;
        }
        d0 = ((s0[0] + s0[1]) + (s0[2] + s0[3])) + ((s0[4] + s0[5]) + (s0[6] + s0[7]));
        d1 = ((s1[0] + s1[1]) + (s1[2] + s1[3])) + ((s1[4] + s1[5]) + (s1[6] + s1[7]));
    }
    for (uint k = 0; k < KSEL; k++) {
        const float wk = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wl), k));
        acc0 += wk * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d0), k));
        acc1 += wk * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(d1), k));
    }
    if (lane == 0) {
        y[(size_t)t * N + row0] = acc0;
        if (two) y[(size_t)t * N + row0 + 1u] = acc1;
    }
}
extern "C" __global__ void __launch_bounds__(256)
moe_down_q4k_dec(const float* act, const uchar* wd, const uint* idx, const float* wgt, float* y, uint K, uint N,
                 uint KSEL, uint E, uint ACC) {
    moe_down_dec_body<W4k, false>(act, wd, idx, wgt, y, K, N, KSEL, E, ACC);
}
extern "C" __global__ void __launch_bounds__(256)
moe_down_q4k_slots(const float* act, const uchar* arena, const unsigned long* off_d, const float* wgt, float* y, uint K,
                   uint N, uint KSEL, uint LIM, uint ACC) {
    moe_down_dec_body<W4k, true>(act, arena, off_d, wgt, y, K, N, KSEL, LIM, ACC);
}
extern "C" __global__ void __launch_bounds__(256)
moe_down_q5k_dec(const float* act, const uchar* wd, const uint* idx, const float* wgt, float* y, uint K, uint N,
                 uint KSEL, uint E, uint ACC) {
    moe_down_dec_body<W5k, false>(act, wd, idx, wgt, y, K, N, KSEL, E, ACC);
}
extern "C" __global__ void __launch_bounds__(256)
moe_down_q6k_dec(const float* act, const uchar* wd, const uint* idx, const float* wgt, float* y, uint K, uint N,
                 uint KSEL, uint E, uint ACC) {
    moe_down_dec_body<W6k, false>(act, wd, idx, wgt, y, K, N, KSEL, E, ACC);
}

// ------------------------------------------------------------------ the quantizer and the grouping in one launch
//   moe_quant_group(x, xq, xs, idx, counts, offsets, list, K, T, NA, E)   grid [T + 1,1,1]: block t quantizes token t
//       (quant_q8k's rule, the operations of quantize_q8k), the last block sorts the assignments by expert (moe_group).
// Neither depends on the other; both are a few microseconds of launch and little else.
extern "C" __global__ void __launch_bounds__(256)
moe_quant_group(const float* __restrict__ x, signed char* __restrict__ xq, float* __restrict__ xs, const uint* __restrict__ idx,
                uint* __restrict__ counts, uint* __restrict__ offsets, uint* __restrict__ list, uint K, uint T, uint NA, uint E) {
    __shared__ uint cnt[1024];
    __shared__ uint off[1025];
    if (blockIdx.x >= T) {
        moe_group_body(idx, counts, offsets, list, NA, E, cnt, off);
        return;
    }
    const size_t t = blockIdx.x;
    block_quant_q8k(x + t * K, K, xq + t * K, xs + t * (K >> 8));
}

// ------------------------------------------------------------------ the router and the quantizer in one launch
//   moe_topk_quant(lg, idx, wgt, x, xq, xs, E, KSEL, K)     grid [tokens,1,1] x 512
// Wave 0 routes the workgroup's token (moe_topk_m's bits) while the others quantize it (quantize_q8k's): a launch less for
// batches whose expert products find their assignments in idx themselves.
extern "C" __global__ void __launch_bounds__(512)
moe_topk_quant(const float* __restrict__ lg, uint* __restrict__ idx, float* __restrict__ wgt, const float* __restrict__ x,
               signed char* __restrict__ xq, float* __restrict__ xs, uint E, uint KSEL, uint K) {
    const size_t t = blockIdx.x;
    if (threadIdx.x < 64u) moe_topk_body(lg + t * E, idx + t * KSEL, wgt + t * KSEL, E, KSEL);
    else block_quant_q8k(x + t * K, K, xq + t * K, xs + t * (K >> 8), 64u, 448u);
}

// ------------------------------------------------------------------ grouped integer dots that find their assignments
//   moe_gu_q4k_mi(xq, xs, wg, wu, act, idx, K, N, KSEL, NA, E)        grid [ceil(N / 8), min(E, NA), 1] x 256; ceil(N / 16) for K <= 1024;
//   moe_gu_q4k_mil(the same)                                          K <= 2048, beyond that _mil
//   moe_down_{q4k,q5k,q6k}_mi(act, wd, dv, idx, K, N, NA, E)          grid [ceil(N / R), min(E, NA), 1] x 256, K <= 2048;
//                                                                     R = 64 for K <= 512, 32 for K <= 1024, else 16
// The _m entries' products and sums, bit for bit, over at most MI_MOST assignments as the router leaves them.  Workgroup y serves
// expert y, or with fewer assignments than experts the expert of assignment y if no earlier one has it: what finds its
// expert's assignments is one load or a few of idx, no launch, and at 4 tokens a quarter of 128 experts' workgroups is
// launched.  The down entries quantize the f32 activations they need into LDS (quantize_q8k's operations), MI_STAGE codes at a time.
// A row of up to 1024 (512) weights takes half (a quarter of) the lanes, so the wave holds two (four) rows side by side; a
// longer one than 2048 is walked with four assignments' sums beside it, so that their expert's rows are read once and not
// once each.  Whole layer: 96 experts of 768 x 2816 at 16 tokens 92.9 -> 85.6 us, of 512 x 1536 (Q6_K down) at 8 26.6 -> 19.6,
// 64 of 512 x 1024 (Q5_K down) at 16 28.1 -> 20.8.
#define MI_MOST 512u
// The expert's assignments as a bit each, in scalar registers: found by every wave for itself, no LDS and no barrier.
template <uint NQ>
struct MiFound {
    uint e;
    unsigned long long m[NQ];
    __device__ __forceinline__ uint count() const {
        uint n = 0u;
#pragma unroll
        for (uint q = 0; q < NQ; q++) n += (uint)__popcll(m[q]);
        return n;
    }
    // the first of those left, taken out of them
    __device__ __forceinline__ uint next() {
        uint a = 0u;
        bool got = false;
#pragma unroll
        for (uint q = 0; q < NQ; q++)
            if (!got && m[q]) {
                a = 64u * q + (uint)__builtin_ctzll(m[q]);
                m[q] &= m[q] - 1ull;
                got = true;
            }
        return a;
    }
};
template <uint NQ>
__device__ __forceinline__ MiFound<NQ> mi_find(const uint* __restrict__ idx, uint NA, uint E) {
    const uint y = blockIdx.y, lane = threadIdx.x & 63u;
    const bool by_a = NA < E;
    uint v[NQ];
#pragma unroll
    for (uint q = 0; q < NQ; q++) v[q] = 64u * q < NA ? idx[min(lane + 64u * q, NA - 1u)] : 0u;
#pragma unroll
    for (uint q = 0; q < NQ; q++) v[q] = lane + 64u * q < NA ? min(v[q], E - 1u) : 0xFFFFFFFFu;   // (as moe_group)
    MiFound<NQ> f;
    f.e = by_a ? min((uint)__builtin_amdgcn_readfirstlane((int)idx[y]), E - 1u) : y;
    bool first = true;
#pragma unroll
    for (uint q = 0; q < NQ; q++) {
        f.m[q] = __ballot(v[q] == f.e);
        if (by_a && 64u * q <= y && (f.m[q] & (y - 64u * q < 64u ? (1ull << (y - 64u * q)) - 1ull : ~0ull))) first = false;
    }
    if (!first) {
#pragma unroll
        for (uint q = 0; q < NQ; q++) f.m[q] = 0ull;
    }
    return f;
}

// G groups of eight lanes per row (eight: the wave's, four: a half's); LONG: rows of more super-blocks than that
template <int G, bool LONG, uint NQ>
__device__ __forceinline__ void moe_gu_mi_body(const signed char* __restrict__ xq, const float* __restrict__ xs, const uchar* __restrict__ wg,
                                               const uchar* __restrict__ wu, float* __restrict__ act, uint K, uint N, uint KSEL, MiFound<NQ> found) {
    const uint e = found.e, n = found.count();
    if (!n) return;
    const uint lane = threadIdx.x & 63u, part = lane / (8u * G), span = 8u * G;
    const uint row0 = ((blockIdx.x * 4u + (threadIdx.x >> 6)) * (64u / span) + part) * 2u;
    const uint nsb = K >> 8, g = (lane >> 3) % G, l = lane & 7u, c = l >> 1;
    const size_t rb = (size_t)nsb * Q4K_BYTES;
    const uint rowc = min(row0, N - 1u);
    const size_t r1 = rowc + 1u < N ? rb : 0;
    const uchar* g0 = wg + ((size_t)e * N + rowc) * rb;
    const uchar* u0 = wu + ((size_t)e * N + rowc) * rb;
    auto store = [&](uint a, float vg0, float vg1, float vu0, float vu1) {
        // the four sums in one pass: lanes 0 / 1 end with the gate sums of the two rows, lanes 2 / 3 with the up sums
        float tot = row16_sum4(vg0, vg1, vu0, vu1, lane);
        tot += __shfl_xor(tot, 16);
        if (G == 8) tot += __shfl_xor(tot, 32);
        const float upv = dpp_f32<OJK_DPP_QUAD_XOR2>(tot);
        const uint j = lane % span;
        if (j < 2u && row0 + j < N) act[(size_t)a * N + row0 + j] = (tot / (1.0f + expf(-tot))) * upv;
    };
    if constexpr (!LONG) {
        const bool on = g < nsb;
        const size_t o = (size_t)(on ? g : 0u) * Q4K_BYTES, oq = o + 16u + l * 16u;
        const uint4 hg0 = *(const uint4*)(g0 + o), qg0 = *(const uint4*)(g0 + oq), hg1 = *(const uint4*)(g0 + r1 + o), qg1 = *(const uint4*)(g0 + r1 + oq);
        const uint4 hu0 = *(const uint4*)(u0 + o), qu0 = *(const uint4*)(u0 + oq), hu1 = *(const uint4*)(u0 + r1 + o), qu1 = *(const uint4*)(u0 + r1 + oq);
#pragma unroll 1
        for (uint i = 0; i < n; i++) {
            const uint a = found.next(), t = a / KSEL;
            Q4kFrag f = q4k_load_frag(xq + (size_t)t * nsb * 256u, xs + (size_t)t * nsb, on ? g : 0u, l);
            f.sx = on ? f.sx : 0.0f;        // (lanes past the row's last super-block: products of zero, no branches)
            store(a, q4k_lane_dot(hg0, qg0, c, f), q4k_lane_dot(hg1, qg1, c, f), q4k_lane_dot(hu0, qu0, c, f), q4k_lane_dot(hu1, qu1, c, f));
        }
        return;
    }
    auto walk = [&](auto m_) {
        constexpr int M = decltype(m_)::value;
        float v[M][4] = {};
        uint a[M], t[M];
#pragma unroll
        for (int k = 0; k < M; k++) a[k] = found.next(), t[k] = a[k] / KSEL;
#pragma unroll 1
        for (uint sb = g; sb < nsb; sb += (uint)G) {
            const size_t o = (size_t)sb * Q4K_BYTES, oq = o + 16u + l * 16u;
            const uint4 hg0 = *(const uint4*)(g0 + o), qg0 = *(const uint4*)(g0 + oq), hg1 = *(const uint4*)(g0 + r1 + o), qg1 = *(const uint4*)(g0 + r1 + oq);
            const uint4 hu0 = *(const uint4*)(u0 + o), qu0 = *(const uint4*)(u0 + oq), hu1 = *(const uint4*)(u0 + r1 + o), qu1 = *(const uint4*)(u0 + r1 + oq);
#pragma unroll
            for (int k = 0; k < M; k++) {
                const Q4kFrag f = q4k_load_frag(xq + (size_t)t[k] * nsb * 256u, xs + (size_t)t[k] * nsb, sb, l);
                v[k][0] += q4k_lane_dot(hg0, qg0, c, f);
                v[k][1] += q4k_lane_dot(hg1, qg1, c, f);
                v[k][2] += q4k_lane_dot(hu0, qu0, c, f);
                v[k][3] += q4k_lane_dot(hu1, qu1, c, f);
            }
        }
#pragma unroll
        for (int k = 0; k < M; k++) store(a[k], v[k][0], v[k][1], v[k][2], v[k][3]);
    };
    uint left = n;
    for (; left >= 4u; left -= 4u) walk(std::integral_constant<int, 4>());
    if (left == 3u) walk(std::integral_constant<int, 3>());
    else if (left == 2u) walk(std::integral_constant<int, 2>());
    else if (left == 1u) walk(std::integral_constant<int, 1>());
}
extern "C" __global__ void __launch_bounds__(256)
moe_gu_q4k_mi(const signed char* __restrict__ xq, const float* __restrict__ xs, const uchar* __restrict__ wg,
              const uchar* __restrict__ wu, float* __restrict__ act, const uint* __restrict__ idx, uint K, uint N, uint KSEL, uint NA, uint E) {
    if (NA <= 128u) {
        const MiFound<2> f = mi_find<2>(idx, NA, E);
        if (K <= 1024u) moe_gu_mi_body<4, false>(xq, xs, wg, wu, act, K, N, KSEL, f);
        else moe_gu_mi_body<8, false>(xq, xs, wg, wu, act, K, N, KSEL, f);
    } else {
        const MiFound<MI_MOST / 64u> f = mi_find<MI_MOST / 64u>(idx, NA, E);
        if (K <= 1024u) moe_gu_mi_body<4, false>(xq, xs, wg, wu, act, K, N, KSEL, f);
        else moe_gu_mi_body<8, false>(xq, xs, wg, wu, act, K, N, KSEL, f);
    }
}
// (an entry of its own: its registers would halve the waves of the other)
extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
moe_gu_q4k_mil(const signed char* __restrict__ xq, const float* __restrict__ xs, const uchar* __restrict__ wg,
               const uchar* __restrict__ wu, float* __restrict__ act, const uint* __restrict__ idx, uint K, uint N, uint KSEL, uint NA, uint E) {
    if (NA <= 128u) moe_gu_mi_body<8, true>(xq, xs, wg, wu, act, K, N, KSEL, mi_find<2>(idx, NA, E));
    else moe_gu_mi_body<8, true>(xq, xs, wg, wu, act, K, N, KSEL, mi_find<MI_MOST / 64u>(idx, NA, E));
}

#define MI_STAGE 8192u
template <class W, int G, uint NQ>
__device__ __forceinline__ void moe_down_mi_body(const float* __restrict__ act, const uchar* __restrict__ wd, float* __restrict__ dv, uint K, uint N,
                                                 MiFound<NQ> found, signed char* lq, float* ls) {
    uint n = found.count();
    if (!n) return;
    const uint tid = threadIdx.x, lane = tid & 63u, span = 8u * G;
    const uint row0 = ((blockIdx.x * 4u + (tid >> 6)) * (64u / span) + lane / span) * 4u, rowc = min(row0, N - 1u);
    const uint nsb = K >> 8, g = (lane >> 3) % G, l = lane & 7u, c = l >> 1;
    const bool on = g < nsb;
    const size_t rb = (size_t)nsb * W::BYTES;
    const uchar* const w0 = wd + ((size_t)found.e * N + rowc) * rb + (size_t)(on ? g : 0u) * W::BYTES;
    W wr[4];
#pragma unroll
    for (uint r = 0; r < 4u; r++) wr[r].load(w0 + (size_t)min(r, N - 1u - rowc) * rb, l);      // on their way while the activations are quantized
    const uint most = MI_STAGE / K;
    for (bool again = false; n; again = true) {
        const uint m = min(most, n);
        MiFound<NQ> q = found;
        if (again) __syncthreads();
        for (uint t = 0; t < m; t++) {
            const float* const p = act + (size_t)q.next() * K;
            for (uint o = tid * 8u; o < K; o += 2048u) {
                float scale;
                *(uint2*)(lq + t * K + o) = oct_quant_q8k(*(const float4*)(p + o), *(const float4*)(p + o + 4), scale);
                if ((tid & 31u) == 0u) ls[t * nsb + (o >> 8)] = scale;
            }
        }
        __syncthreads();
#pragma unroll 1
        for (uint t = 0; t < m; t++) {
            const uint a = found.next();
            Q4kFrag f = q4k_load_frag(lq + t * K, ls + t * nsb, on ? g : 0u, l);
            f.sx = on ? f.sx : 0.0f;
            float v = row16_sum4(wr[0].dot(c, f), wr[1].dot(c, f), wr[2].dot(c, f), wr[3].dot(c, f), lane);
            if (G >= 4) v += __shfl_xor(v, 16);
            if (G == 8) v += __shfl_xor(v, 32);
            const uint j = lane % span;
            if (j < 4u && row0 + j < N) dv[(size_t)a * N + row0 + j] = v;
        }
        n -= m;
    }
}
template <class W, uint NQ>
__device__ __forceinline__ void moe_down_mi_pick(const float* __restrict__ act, const uchar* __restrict__ wd, float* __restrict__ dv, uint K, uint N,
                                                 const MiFound<NQ>& f, signed char* lq, float* ls) {
    if (K <= 512u) moe_down_mi_body<W, 2>(act, wd, dv, K, N, f, lq, ls);
    else if (K <= 1024u) moe_down_mi_body<W, 4>(act, wd, dv, K, N, f, lq, ls);
    else moe_down_mi_body<W, 8>(act, wd, dv, K, N, f, lq, ls);
}
#define MOE_DOWN_MI(FMT, W)                                                                                                  \
    extern "C" __global__ void __launch_bounds__(256)                                                                       \
    moe_down_##FMT##_mi(const float* __restrict__ act, const uchar* __restrict__ wd, float* __restrict__ dv,                 \
                        const uint* __restrict__ idx, uint K, uint N, uint NA, uint E) {                                     \
        __shared__ __align__(16) signed char lq[MI_STAGE];                                                                   \
        __shared__ float ls[MI_STAGE / 256u];                                                                                \
        if (NA <= 128u) moe_down_mi_pick<W>(act, wd, dv, K, N, mi_find<2>(idx, NA, E), lq, ls);                              \
        else moe_down_mi_pick<W>(act, wd, dv, K, N, mi_find<MI_MOST / 64u>(idx, NA, E), lq, ls);                                         \
    }
MOE_DOWN_MI(q4k, W4k)
MOE_DOWN_MI(q5k, W5k)
MOE_DOWN_MI(q6k, W6k)

// ------------------------------------------------------------------ Q8_0 experts, f32 activations
//   moe_gu_q80(x, wg, wu, act, idx, K, N)              grid [ceil(N/8), KSEL, tokens], block 256
//   moe_down_q80(act, wd, y, idx, wgt, K, N, KSEL)     grid [1 .. ceil(N/4), tokens, 1], block 256 (rows grid-stride,
//                                                      4 per workgroup and step: the reference's ceil(N/32) is a valid grid)
// The reference's expert kernels by their own names and arguments
// (crates/ojas-cuda/src/kernels/moe.rs:75-125): act[j][n] = silu(gate_e . x) * (up_e . x) for the expert
// e = idx[j] of slot j, and y[n] += sum_j wgt[j] * (down_e . act[j]) — the down launch accumulates onto y.  Q8_0 rows meet f32 activations, as dot_q80 does
// (crates/ojas-cpu/src/cpu_math.rs:971-981).  The third (second) grid dimension walks tokens: token t
// reads x + t K, idx + t KSEL, wgt + t KSEL and writes act + t KSEL N, y + t N; a one-token caller
// leaves it at 1.  Four lanes share a 34-byte block, a wave walks 16 blocks per step.  The trailing E is
// not part of the reference's argument list: the dispatcher derives it from the extent of the expert
// tensors, and a slot whose index is E or more contributes zeros rather than reading past them.
__device__ __forceinline__ float q80f_block_part(const uchar* blk, uint p, float4 x0, float4 x1) {
    const u32x2_a2 q = *(const u32x2_a2*)(blk + 2u + p * 8u);
    float a = (float)(signed char)(q.x) * x0.x;
    a = fmaf((float)(signed char)(q.x >> 8), x0.y, a);
    a = fmaf((float)(signed char)(q.x >> 16), x0.z, a);
    a = fmaf((float)((int)q.x >> 24), x0.w, a);
    a = fmaf((float)(signed char)(q.y), x1.x, a);
    a = fmaf((float)(signed char)(q.y >> 8), x1.y, a);
    a = fmaf((float)(signed char)(q.y >> 16), x1.z, a);
    a = fmaf((float)((int)q.y >> 24), x1.w, a);
    return f16_bits_to_f32(*(const ushort*)blk) * a;
}

// gate/up rows of one expert (eg, eu: its first rows) against token row xt; nb = 0 skips the products
__device__ __forceinline__ void moe_gu_q80_body(const float* __restrict__ xt, const uchar* __restrict__ eg,
                                                const uchar* __restrict__ eu, float* __restrict__ act_row,
                                                uint K, uint N, uint nb) {
    const uint lane = threadIdx.x & 63u, g = lane >> 2, p = lane & 3u;
    const uint row0 = (blockIdx.x * 4u + (threadIdx.x >> 6)) * 2u;
    if (row0 >= N) return;
    const size_t rb = (size_t)(K >> 5) * Q80_BYTES;
    float ag[2] = {0.0f, 0.0f}, au[2] = {0.0f, 0.0f};
    for (uint b = g; b < nb; b += 16u) {
        const float4* xp = (const float4*)(xt + (size_t)b * 32u + p * 8u);
        const float4 x0 = xp[0], x1 = xp[1];
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const size_t off = (size_t)min(row0 + (uint)r, N - 1u) * rb + (size_t)b * Q80_BYTES;
            ag[r] += q80f_block_part(eg + off, p, x0, x1);
            au[r] += q80f_block_part(eu + off, p, x0, x1);
        }
    }
#pragma unroll
    for (int r = 0; r < 2; r++) {
        const float gs = wave_sum(ag[r]), us = wave_sum(au[r]);
        if (lane == 0 && row0 + r < N) act_row[row0 + r] = (gs / (1.0f + expf(-gs))) * us;
    }
}

// four down rows of one expert (ed: its first row) against one activation row
__device__ __forceinline__ void moe_down_q80_part(const float* __restrict__ xr, const uchar* __restrict__ ed,
                                                  uint K, uint N, uint row0, float wj, float (&res)[4]) {
    const uint lane = threadIdx.x & 63u, g = lane >> 2, p = lane & 3u;
    const uint nb = K >> 5;
    const size_t rb = (size_t)nb * Q80_BYTES;
    float a[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    for (uint b = g; b < nb; b += 16u) {
        const float4* xp = (const float4*)(xr + (size_t)b * 32u + p * 8u);
        const float4 x0 = xp[0], x1 = xp[1];
#pragma unroll
        for (int r = 0; r < 4; r++)
            a[r] += q80f_block_part(ed + (size_t)min(row0 + (uint)r, N - 1u) * rb + (size_t)b * Q80_BYTES, p, x0, x1);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) res[r] += wj * wave_sum(a[r]);
}

extern "C" __global__ void __launch_bounds__(256)
moe_gu_q80(const float* __restrict__ x, const uchar* __restrict__ wg, const uchar* __restrict__ wu,
           float* __restrict__ act, const uint* __restrict__ idx, uint K, uint N, uint E) {
    const uint j = blockIdx.y, t = blockIdx.z, ksel = gridDim.y;
    const uint e = idx[t * ksel + j];
    const size_t eb = (size_t)(e < E ? e : 0u) * N * ((size_t)(K >> 5) * Q80_BYTES);
    moe_gu_q80_body(x + (size_t)t * K, wg + eb, wu + eb, act + ((size_t)t * ksel + j) * N, K, N, e < E ? K >> 5 : 0u);
}

// The down launches: a workgroup owns four rows at a time (rows grid-stride over the workgroups), its four
// waves take the slots j = wave, wave + 4, ... and meet in LDS, where the partial sums are added in wave order
// onto y — an expert row is short (a few hundred to a few thousand weights), so the slots are the parallelism
// that fills the chip at one token.
__device__ __forceinline__ void moe_down_finish(float (&res)[4], float* __restrict__ yt, uint N, uint row0) {
    __shared__ float part[4][4];
    const uint lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < 4; r++) part[wave][r] = res[r];
    }
    __syncthreads();
    if (threadIdx.x < 4u && row0 + threadIdx.x < N)
        yt[row0 + threadIdx.x] += ((part[0][threadIdx.x] + part[1][threadIdx.x]) + part[2][threadIdx.x]) + part[3][threadIdx.x];
    __syncthreads();
}

extern "C" __global__ void __launch_bounds__(256)
moe_down_q80(const float* __restrict__ act, const uchar* __restrict__ wd, float* __restrict__ y,
             const uint* __restrict__ idx, const float* __restrict__ wgt, uint K, uint N, uint KSEL, uint E) {
    const uint t = blockIdx.y, wave = threadIdx.x >> 6;
    const size_t eb = (size_t)N * ((size_t)(K >> 5) * Q80_BYTES);
    for (uint row0 = blockIdx.x * 4u; row0 < N; row0 += gridDim.x * 4u) {
        float res[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint j = wave; j < KSEL; j += 4u) {
            const uint e = idx[t * KSEL + j];
            if (e >= E) continue;
            moe_down_q80_part(act + ((size_t)t * KSEL + j) * K, wd + (size_t)e * eb, K, N, row0, wgt[t * KSEL + j], res);
        }
        moe_down_finish(res, y + (size_t)t * N, N, row0);
    }
}

// Streamed Q8_0 experts (crates/ojas-cuda/src/kernels/moe.rs:133-174): the experts of a layer sit at whatever
// slots of a cache arena were free, and the host passes one u32 byte offset per selected expert in place of
// the index.   moe_gu_q80_slots(x, arena_g, arena_u, act, off_g, off_u, K, N)   grid [ceil(N/8), KSEL, tokens]
//              moe_down_q80_slots(act, arena, y, off_d, wgt, K, N, KSEL)          grid [1 .. ceil(N/4), tokens, 1]
// The trailing LIM constants are appended by the dispatcher — the last offset at which a whole expert still
// fits its arena — and an offset is rounded down to the blocks' two-byte alignment and clamped to LIM, so a bad
// table reads a wrong expert, never past the arena.
extern "C" __global__ void __launch_bounds__(256)
moe_gu_q80_slots(const float* __restrict__ x, const uchar* __restrict__ arena_g, const uchar* __restrict__ arena_u,
                 float* __restrict__ act, const uint* __restrict__ off_g, const uint* __restrict__ off_u,
                 uint K, uint N, uint LIM_G, uint LIM_U) {
    const uint j = blockIdx.y, t = blockIdx.z, ksel = gridDim.y;
    const uint og = min(off_g[t * ksel + j] & ~1u, LIM_G), ou = min(off_u[t * ksel + j] & ~1u, LIM_U);
    moe_gu_q80_body(x + (size_t)t * K, arena_g + og, arena_u + ou, act + ((size_t)t * ksel + j) * N, K, N, K >> 5);
}

extern "C" __global__ void __launch_bounds__(256)
moe_down_q80_slots(const float* __restrict__ act, const uchar* __restrict__ arena, float* __restrict__ y,
                   const uint* __restrict__ off_d, const float* __restrict__ wgt, uint K, uint N, uint KSEL, uint LIM) {
    const uint t = blockIdx.y, wave = threadIdx.x >> 6;
    for (uint row0 = blockIdx.x * 4u; row0 < N; row0 += gridDim.x * 4u) {
        float res[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint j = wave; j < KSEL; j += 4u)
            moe_down_q80_part(act + ((size_t)t * KSEL + j) * K, arena + min(off_d[t * KSEL + j] & ~1u, LIM), K, N, row0,
                              wgt[t * KSEL + j], res);
        moe_down_finish(res, y + (size_t)t * N, N, row0);
    }
}

// ------------------------------------------------------------------ grouped products on the matrix cores
// A workgroup owns 16 rows of expert e and walks the expert's assignments 16 at a time.  Per 32-weight
// sub-block one v_mfma_i32_16x16x32_i8 multiplies the tile of quantized activations (A: lane
// (m, kg) = (lane % 16, lane / 16) holds bytes 8 kg .. 8 kg + 7 of token m) with the sub-block's
// 4-bit codes as bytes (B: lane (n, kg) holds the same bytes of row n); D register v of lane
// (n, kg) is the integer dot of token 4 kg + v with row n.  A second MFMA against a tile of ones
// gives every lane the activations' sub-block sums in the same layout, so the scale algebra
//     sum_sb sx[t][sb] * ( d * sum_j sc_j * idot_j  -  dmin * sum_j m_j * bsum_j )
// needs no cross-lane traffic: per MFMA result register one integer multiply-add with a
// lane-constant 6-bit scale (the sums over j are exact in int32: |.| < 2^25), and per super-block
// two converts and three FMAs, the form of dot_q4k itself (crates/ojas-cpu/src/cpu_math.rs:609-635).  A token's result does not
// depend on which other tokens share its tile.
typedef int int4v __attribute__((ext_vector_type(4)));

__device__ __forceinline__ long pack2(uint lo, uint hi) { return (long)(((unsigned long)hi << 32) | lo); }

// acc[w][v] += sx[v] * sum_j (a_j * idot_j[v] - b_j * bsum_j[v]) for one super-block of NW weight
// tensors sharing the activations.  `xsb` points at the lane's 8 bytes of sub-block 0 (sub-block j
// 32 bytes further); `wblk[w]` at the lane's row inside a wave-private LDS copy of the 16 x 144-byte
// tile.
template <int NW>
__device__ __forceinline__ void mm_superblock(const signed char* xsb, const uchar* const (&wblk)[NW], uint kg,
                                              const float (&sx)[4], float (&acc)[NW][4]) {
    // integer partial sums are exact, so sum_j sc_j * idot_j and sum_j m_j * bsum_j are formed in
    // int32 (one v_mad_i32_i24 per MFMA result register) and converted once per super-block
    int isum[NW][4], msum[NW][4];
    float d[NW], dmin[NW];
    uint s0[NW], s1[NW], s2[NW];
#pragma unroll
    for (int w = 0; w < NW; w++) {
        const uint4 hdr = *(const uint4*)wblk[w];
        d[w] = f16_bits_to_f32(hdr.x & 0xFFFFu);
        dmin[w] = f16_bits_to_f32(hdr.x >> 16);
        s0[w] = hdr.y; s1[w] = hdr.z; s2[w] = hdr.w;
#pragma unroll
        for (int v = 0; v < 4; v++) { isum[w][v] = 0; msum[w][v] = 0; }
    }
    const long ones = 0x0101010101010101L;
    const int4v zero = {0, 0, 0, 0};
    // (kept rolled: unrolled, the compiler holds every scale and code of the super-block at once,
    // occupancy drops, and the kernel measured slower)
#pragma unroll 1
    for (uint c = 0; c < 4u; c++) {
        const uint2 x0 = *(const uint2*)(xsb + c * 64u), x1 = *(const uint2*)(xsb + c * 64u + 32u);
        const long A0 = pack2(x0.x, x0.y), A1 = pack2(x1.x, x1.y);
        const int4v b0 = __builtin_amdgcn_mfma_i32_16x16x32_i8(A0, ones, zero, 0, 0, 0);
        const int4v b1 = __builtin_amdgcn_mfma_i32_16x16x32_i8(A1, ones, zero, 0, 0, 0);
#pragma unroll
        for (int w = 0; w < NW; w++) {
            uint sc, mn;
            q4k_scale_min_pair(s0[w], s1[w], s2[w], c, sc, mn);
            const int sc_lo = (int)(sc & 0xFFu), sc_hi = (int)(sc >> 8), m_lo = (int)(mn & 0xFFu), m_hi = (int)(mn >> 8);
            const uint2 q = *(const uint2*)(wblk[w] + 16u + c * 32u + 8u * kg);
            const int4v dl = __builtin_amdgcn_mfma_i32_16x16x32_i8(A0, pack2(q.x & 0x0F0F0F0Fu, q.y & 0x0F0F0F0Fu), zero, 0, 0, 0);
            const int4v dh = __builtin_amdgcn_mfma_i32_16x16x32_i8(A1, pack2((q.x >> 4) & 0x0F0F0F0Fu, (q.y >> 4) & 0x0F0F0F0Fu), zero, 0, 0, 0);
#pragma unroll
            for (int v = 0; v < 4; v++) {
                isum[w][v] += __mul24(sc_lo, dl[v]) + __mul24(sc_hi, dh[v]);
                msum[w][v] += __mul24(m_lo, b0[v]) + __mul24(m_hi, b1[v]);
            }
        }
    }
#pragma unroll
    for (int w = 0; w < NW; w++)
#pragma unroll
        for (int v = 0; v < 4; v++) acc[w][v] += sx[v] * (d[w] * (float)isum[w][v] - dmin[w] * (float)msum[w][v]);
}

// Copy the super-block `sb` of 16 consecutive rows (144 bytes each, `rb` apart, rows past `nrows`
// clamped) into the wave's LDS tile with 16-byte pieces, 64 lanes side by side: the loads are
// contiguous per row instead of 8 bytes per lane and row.
__device__ __forceinline__ void mm_stage_tile(const uchar* w_row0, size_t rb, uint nrows, uint sb, uchar* tile, uint lane) {
#pragma unroll
    for (int i = 0; i < 3; i++) {
        const uint p = lane + 64u * i;
        if (p < 144u) {
            const uint r = p / 9u, c = p - r * 9u;
            *(uint4*)(tile + p * 16u) = *(const uint4*)(w_row0 + (size_t)min(r, nrows - 1u) * rb + (size_t)sb * Q4K_BYTES + c * 16u);
        }
    }
}

// Workgroup = one 16-row tile of expert e; its four waves split the super-blocks of K between
// them (wave w takes w, w + 4, ...) and their partial sums meet in LDS, added in wave order.
template <int NW>
__device__ __forceinline__ void mm_reduce(float (&acc)[NW][4], float* red, uint wave, uint lane) {
    // red: [3 waves][NW * 4][64 lanes]
    if (wave > 0) {
#pragma unroll
        for (int w = 0; w < NW; w++)
#pragma unroll
            for (int v = 0; v < 4; v++) red[((wave - 1u) * (NW * 4) + w * 4 + v) * 64u + lane] = acc[w][v];
    }
    __syncthreads();
    if (wave == 0) {
#pragma unroll
        for (int k = 0; k < 3; k++)
#pragma unroll
            for (int w = 0; w < NW; w++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[w][v] += red[(k * (NW * 4) + w * 4 + v) * 64u + lane];
    }
    __syncthreads();
}

// (four waves per SIMD: latency of the dependent list -> activation -> weight loads is hidden by occupancy)
extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
moe_gu_q4k_mm(const signed char* __restrict__ xq, const float* __restrict__ xs, const uchar* __restrict__ wg,
              const uchar* __restrict__ wu, float* __restrict__ act, const uint* __restrict__ offsets,
              const uint* __restrict__ list, uint K, uint N, uint KSEL, uint NA) {
    __shared__ float red[3 * 8 * 64];
    __shared__ __attribute__((aligned(16))) uchar tiles[4][2][16 * Q4K_BYTES];
    const uint e = blockIdx.y;
    const uint a0 = min(offsets[e], NA), a1 = min(offsets[e + 1], NA);
    if (a0 >= a1) return;
    const uint lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, n = lane & 15u, kg = lane >> 4;
    const uint row0 = blockIdx.x * 16u;
    const uint nsb = K >> 8;
    const size_t rb = (size_t)nsb * Q4K_BYTES;
    const uchar* gw = wg + ((size_t)e * N + row0) * rb;
    const uchar* uw = wu + ((size_t)e * N + row0) * rb;
    const uint nrows = min(16u, N - row0);
    for (uint tt = a0; tt < a1; tt += 16u) {
        // activations: lane's token for the A operand, and the four tokens of its D registers
        const uint ta = min(list[min(tt + n, a1 - 1u)], NA - 1u) / KSEL;
        const signed char* xrow = xq + (size_t)ta * K + 8u * kg;
        uint av[4], tv[4];
#pragma unroll
        for (int v = 0; v < 4; v++) {
            av[v] = min(list[min(tt + 4u * kg + v, a1 - 1u)], NA - 1u);
            tv[v] = av[v] / KSEL;
        }
        float acc[2][4];
#pragma unroll
        for (int w = 0; w < 2; w++)
#pragma unroll
            for (int v = 0; v < 4; v++) acc[w][v] = 0.0f;
#pragma unroll 1
        for (uint sb = wave; sb < nsb; sb += 4u) {
            float sx[4];
#pragma unroll
            for (int v = 0; v < 4; v++) sx[v] = xs[(size_t)tv[v] * nsb + sb];
            mm_stage_tile(gw, rb, nrows, sb, tiles[wave][0], lane);
            mm_stage_tile(uw, rb, nrows, sb, tiles[wave][1], lane);
            const uchar* const wb[2] = {tiles[wave][0] + n * Q4K_BYTES, tiles[wave][1] + n * Q4K_BYTES};
            mm_superblock<2>(xrow + sb * 256u, wb, kg, sx, acc);
        }
        mm_reduce<2>(acc, red, wave, lane);
        if (wave == 0 && row0 + n < N) {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (tt + 4u * kg + v < a1) {
                    const float g = acc[0][v];
                    act[(size_t)av[v] * N + row0 + n] = (g / (1.0f + expf(-g))) * acc[1][v];
                }
        }
    }
}

extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 8)))
moe_down_q4k_mm(const signed char* __restrict__ aq, const float* __restrict__ as_, const uchar* __restrict__ wd,
                float* __restrict__ dv, const uint* __restrict__ offsets, const uint* __restrict__ list,
                uint K, uint N, uint NA) {
    __shared__ float red[3 * 4 * 64];
    __shared__ __attribute__((aligned(16))) uchar tiles[4][16 * Q4K_BYTES];
    const uint e = blockIdx.y;
    const uint a0 = min(offsets[e], NA), a1 = min(offsets[e + 1], NA);
    if (a0 >= a1) return;
    const uint lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, n = lane & 15u, kg = lane >> 4;
    const uint row0 = blockIdx.x * 16u;
    const uint nsb = K >> 8;
    const size_t rb = (size_t)nsb * Q4K_BYTES;
    const uchar* dw = wd + ((size_t)e * N + row0) * rb;
    const uint nrows = min(16u, N - row0);
    for (uint tt = a0; tt < a1; tt += 16u) {
        const uint aa = min(list[min(tt + n, a1 - 1u)], NA - 1u);
        const signed char* xrow = aq + (size_t)aa * K + 8u * kg;
        uint av[4];
#pragma unroll
        for (int v = 0; v < 4; v++) av[v] = min(list[min(tt + 4u * kg + v, a1 - 1u)], NA - 1u);
        float acc[1][4] = {{0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll 1
        for (uint sb = wave; sb < nsb; sb += 4u) {
            float sx[4];
#pragma unroll
            for (int v = 0; v < 4; v++) sx[v] = as_[(size_t)av[v] * nsb + sb];
            mm_stage_tile(dw, rb, nrows, sb, tiles[wave], lane);
            const uchar* const wb[1] = {tiles[wave] + n * Q4K_BYTES};
            mm_superblock<1>(xrow + sb * 256u, wb, kg, sx, acc);
        }
        mm_reduce<1>(acc, red, wave, lane);
        if (wave == 0 && row0 + n < N) {
#pragma unroll
            for (int v = 0; v < 4; v++)
                if (tt + 4u * kg + v < a1) dv[(size_t)av[v] * N + row0 + n] = acc[0][v];
        }
    }
}

// ------------------------------------------------------------------ grouped products, a wave per row tile
//   moe_gu_q4k_mt / moe_down_q4k_mt (the arguments of the _m entries)   grid [RG, E, 1], block 512 or 1024,
//                                                                       16 (K + 32) + 5 K / 4 + 320 <= 81920
// With many small experts (128 x 768 x 2048) the _mm form spends its time around the products: a
// workgroup per 16-row tile and expert (16384 of them for the down matrices, three super-blocks
// each), activations fetched from global memory per super-block, partial sums of four waves
// through LDS.  Here RG workgroups share an expert: each stages the expert's next assignments
// once (token rows gathered through the list into LDS, scales, sums split into int8 parts; rows
// past the count are one block of zeros), then every wave walks whole row tiles, all of K, and no partial sums meet.
// A gate and an up wave share a tile: the up wave's sums pass through LDS to the gate wave, which writes silu(g) u.
// What bounds it is the stream of weights: copied alone the gate/up launch (128 experts of 768 x 2048, 2048 assignments,
// 226 MB) takes 48 us and 9 of them are the launch and the staging.  So the rows travel global -> LDS by
// global_load_lds_dwordx4 (nine lanes per row, two units of 16 rows x one super-block in flight per wave, sixteen waves:
// 74 KB per CU) instead of by loads into registers, whose 8-byte pieces of sixteen far-apart rows kept the address unit
// busy; and a super-block's scales are folded into two int8 planes once for all its passes (gq_planes) instead of
// multiplied onto every result.  Eight waves with one tile of both tensors each 68 us, twelve 58, sixteen with a tile of
// both 55 - 59 by how evenly the tiles divide.  Before (loads into registers, gq_superblock): gate/up 81 us, down 46;
// now 58 and 33.  Super-blocks are added in order.
#define MT_LDS 81920u
#define MT_UNIT 2304u
#define MT_DEPTH 2
#define MT_RING (16u * MT_DEPTH * MT_UNIT)
// Down tensors in Q6_K and Q5_K (moe_down_{q6k,q5k}_mt) take the same walk.  Their integers, scale x (code - 32) or scale x
// code, enter as two signed digits (gq_scale4), and their rows, 210 bytes apart or 176, pass through registers: 16-byte
// pieces, neighbouring lanes side by side in a row, one unit ahead, into the wave's own part of LDS and out of it in operand
// order.  Lane (n, kg) holds of row n: Q6_K the 16-position column kg % 2 of the four quarters of half kg / 2; Q5_K positions
// 16 (kg % 2) .. of the sub-blocks of parity kg / 2.
struct MtQ4K {};
struct MtQ6K {
    static constexpr uint BYTES = Q6K_BYTES, PIECES = 13u;
    static constexpr bool MINS = false;
    uint4 a, b, qh;
    uint2 sc;
    uint d16;
    static __device__ __forceinline__ uint tail(const uchar* blk) { return *(const ushort*)(blk + 208u); }
    static __device__ __forceinline__ uint token_at(uint kg) { return 128u * (kg >> 1) + 16u * (kg & 1u); }
    static constexpr uint STEP = 32u;           // a token's bytes of the next instruction
    __device__ __forceinline__ void read(const uchar* row, uint kg, uint d) {
        const uint hf = kg >> 1, h = kg & 1u;
        a = *(const uint4*)(row + 64u * hf + 16u * h);
        b = *(const uint4*)(row + 64u * hf + 32u + 16u * h);
        qh = *(const uint4*)(row + 128u + 32u * hf + 16u * h);
        sc = *(const uint2*)(row + 192u + 8u * hf);
        d16 = d;
    }
    __device__ __forceinline__ void planes(uint kg, gq_i4 (&BH)[4], gq_i4 (&BL)[4]) const {
        const uint s8 = 8u * (kg & 1u), hs[4] = {qh.x, qh.y, qh.z, qh.w};
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const uint4 l = (q & 1) ? b : a;
            const uint ls[4] = {l.x, l.y, l.z, l.w};
            const int s2 = 2 * (int)(signed char)((q < 2 ? sc.x : sc.y) >> (16u * (uint)(q & 1) + s8));
            const ushort bb = (ushort)(128 - 32 * s2);
            const gq_u16x2 f = {(ushort)s2, (ushort)s2}, c = {bb, bb};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint nib = (q & 2) ? ls[i] >> 4 : ls[i];
                const uint two = q == 3 ? hs[i] >> 2 : q == 2 ? hs[i] : q == 1 ? hs[i] << 2 : hs[i] << 4;
                int hi, lo;
                gq_scale4((nib & 0x0F0F0F0Fu) | (two & 0x30303030u), f, c, hi, lo);
                BH[q][i] = hi;
                BL[q][i] = lo;
            }
        }
    }
    __device__ __forceinline__ float d() const { return f16_bits_to_f32(d16); }
    __device__ __forceinline__ float dmin() const { return 0.0f; }
    __device__ __forceinline__ long mins(uint) const { return 0; }
};
struct MtQ5K {
    static constexpr uint BYTES = Q5K_BYTES, PIECES = 11u;
    static constexpr bool MINS = true;
    uint4 hdr, qh, qs[4];
    static __device__ __forceinline__ uint tail(const uchar*) { return 0u; }
    static __device__ __forceinline__ uint token_at(uint kg) { return 16u * kg; }
    static constexpr uint STEP = 64u;
    __device__ __forceinline__ void read(const uchar* row, uint kg, uint) {
        const uint h = 16u * (kg & 1u);
        hdr = *(const uint4*)row;
        qh = *(const uint4*)(row + 16u + h);
#pragma unroll
        for (int c = 0; c < 4; c++) qs[c] = *(const uint4*)(row + 48u + 32u * (uint)c + h);
    }
    __device__ __forceinline__ void planes(uint kg, gq_i4 (&BH)[4], gq_i4 (&BL)[4]) const {
        const uint par = kg >> 1, sc_lo = hdr.y & 0x3F3F3F3Fu, sc_hi = (hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u);
        const uint hs[4] = {qh.x >> par, qh.y >> par, qh.z >> par, qh.w >> par};    // sub-block 2 c + par: bit 2 c
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const uint s2 = 2u * (((c < 2 ? sc_lo : sc_hi) >> (16u * (uint)(c & 1) + 8u * par)) & 0xFFu);
            const gq_u16x2 f = {(ushort)s2, (ushort)s2}, o = {128, 128};
            const uint ls[4] = {qs[c].x, qs[c].y, qs[c].z, qs[c].w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const uint bit = c == 0 ? hs[i] << 4 : c == 1 ? hs[i] << 2 : c == 2 ? hs[i] : hs[i] >> 2;
                int hi, lo;
                gq_scale4(((ls[i] >> (4u * par)) & 0x0F0F0F0Fu) | (bit & 0x10101010u), f, o, hi, lo);
                BH[c][i] = hi;
                BL[c][i] = lo;
            }
        }
    }
    __device__ __forceinline__ float d() const { return f16_bits_to_f32(hdr.x & 0xFFFFu); }
    __device__ __forceinline__ float dmin() const { return f16_bits_to_f32(hdr.x >> 16); }
    __device__ __forceinline__ long mins(uint kg) const {
        const uint mn_lo = hdr.z & 0x3F3F3F3Fu, mn_hi = ((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u);
        return kg == 0u ? gq_pack(mn_lo, mn_hi) : 0;
    }
};
template <class W> struct MtRing { static constexpr uint WAVE = 16u * 16u * W::PIECES + 32u; };      // one unit and its d's
template <> struct MtRing<MtQ4K> { static constexpr uint WAVE = (uint)MT_DEPTH * MT_UNIT; };
template <class W> struct MtBytes { static constexpr uint N = W::BYTES; };
template <> struct MtBytes<MtQ4K> { static constexpr uint N = Q4K_BYTES; };
// One pass of 16 tokens against those digits, as gq_planes_pass
template <class W>
__device__ __forceinline__ void mt_digits_pass(const gq_i4 (&BH)[4], const gq_i4 (&BL)[4], long Bm, float dh, float dmin, const uchar* xp,
                                               const uchar* pq, const float* sx16, uint kg, float (&acc)[4]) {
    const gq_i4 zero = {0, 0, 0, 0};
    gq_i4 DH = zero, DL = zero, Dlo = zero, Dhi = zero;
#pragma unroll
    for (int c = 0; c < 4; c++) {
        const gq_i4 A = *(const gq_i4*)(xp + W::STEP * (uint)c);
        DH = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, BH[c], DH, 0, 0, 0);
        DL = __builtin_amdgcn_mfma_i32_16x16x64_i8(A, BL[c], DL, 0, 0, 0);
    }
    if (W::MINS) {
        const gq_i4 lh = *(const gq_i4*)pq;
        Dlo = __builtin_amdgcn_mfma_i32_16x16x32_i8(gq_pack((uint)lh[0], (uint)lh[1]), Bm, zero, 0, 0, 0);
        Dhi = __builtin_amdgcn_mfma_i32_16x16x32_i8(gq_pack((uint)lh[2], (uint)lh[3]), Bm, zero, 0, 0, 0);
    }
    const float4 sx = *(const float4*)(sx16 + 4u * kg);
    const float sxv[4] = {sx.x, sx.y, sx.z, sx.w};
#pragma unroll
    for (int v = 0; v < 4; v++) {
        const float isum = (float)(DH[v] * 256 + DL[v]);
        acc[v] = W::MINS ? __fmaf_rn(sxv[v], __fmaf_rn(-dmin, (float)(Dhi[v] * 64 + Dlo[v]), __fmul_rn(dh, isum)), acc[v])
                         : __fmaf_rn(__fmul_rn(sxv[v], dh), isum, acc[v]);
    }
}
// What workgroup column y serves, found by the workgroup itself among idx[0 .. NA - 1] (NA <= 4096): with a column per expert
// expert y's assignments; with a column per assignment those of its expert, unless an earlier one has it.  In order: a wave
// scans a run of them, then all know their number and write them to the end of the staging area.  32 integers of LDS at its
// start; a barrier has to pass before those are written over or the list is read.
#define MT_LIST(n) (((n) * 2u + 15u) & ~15u)
struct MtFound { uint e, n; };
__device__ __forceinline__ MtFound mt_find(const uint* __restrict__ idx, uint NA, uint E, uchar* lds) {
    uint* const wt = (uint*)lds;
    const uint lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, nw = blockDim.x >> 6, steps = (NA + 64u * nw - 1u) / (64u * nw);
    const uint first = wave * steps * 64u + lane, y = blockIdx.y;
    const bool by_a = NA < E;
    uint v[8], mine = 0u, ahead = 0u;
#pragma unroll
    for (uint q = 0; q < 8u; q++) v[q] = q < steps && first + 64u * q < NA ? idx[first + 64u * q] : 0xFFFFFFFFu;
    const uint e = by_a ? min((uint)__builtin_amdgcn_readfirstlane((int)idx[y]), E - 1u) : y;
    if (e == E - 1u)        // (only its workgroups clamp what they have loaded, as moe_group does)
#pragma unroll
        for (uint q = 0; q < 8u; q++) v[q] = q < steps && first + 64u * q < NA ? min(v[q], E - 1u) : 0xFFFFFFFFu;
#pragma unroll
    for (uint q = 0; q < 8u; q++) {
        mine += (uint)__popcll(__ballot(v[q] == e));
        if (by_a) ahead += (uint)__popcll(__ballot(v[q] == e && first + 64u * q < y));
    }
    if (lane == 0u) wt[wave] = mine, wt[16u + wave] = ahead;
    __syncthreads();
    uint at = 0u, n = 0u;
    ahead = 0u;
    for (uint w = 0; w < nw; w++) {
        const uint c = wt[w];
        if (w < wave) at += c;
        n += c;
        ahead += wt[16u + w];
    }
    if (ahead) n = 0u;
    n = (uint)__builtin_amdgcn_readfirstlane((int)n);
    if (n) {
        ushort* const lst = (ushort*)(lds + MT_LDS - MT_LIST(n));
#pragma unroll
        for (uint q = 0; q < 8u; q++) {
            const unsigned long long hit = __ballot(v[q] == e);
            if (v[q] == e) lst[at + __builtin_amdgcn_mbcnt_hi((uint)(hit >> 32), __builtin_amdgcn_mbcnt_lo((uint)hit, 0u))] = (ushort)(first + 64u * q);
            at += (uint)__popcll(hit);
        }
    }
    MtFound f;
    f.e = e;
    f.n = n;
    return f;
}
// A pass stages 16 P assignments: as many tiles as the expert has, up to four and to what fits (16 P (K + 32) + 5 P K / 4 + 64 P
// + 256 <= 81920).  An expert's rows are read and unpacked once per pass (2048 x 768, 256 tokens over 128 experts with 8 slots
// each, 16 per expert on average: with one tile of 16 a pass every other expert was read twice; 512 tokens 181 -> 164 us the
// layer with the down rows read once where two tiles read them twice).  A wider pass than the expert fills costs (32 experts
// of 512 x 1536 at 19 each, the layer 36.0 us at the width that fits the count, 37.8 at the widest that fits LDS).
template <class W, bool GU, bool IDX, int P>
__device__ __forceinline__ void moe_mt_body(const signed char* __restrict__ xq, const float* __restrict__ xs,
                                            const uchar* __restrict__ w0, const uchar* __restrict__ w1, float* __restrict__ out,
                                            const uint* __restrict__ offsets, const uint* __restrict__ list,
                                            uint K, uint N, uint KSEL, uint NA, uchar* lds, const MtFound& found) {
    constexpr bool DMA = std::is_same<W, MtQ4K>::value;
    constexpr bool QUANT = IDX && !GU;             // the down entries that find their assignments quantize them too
    constexpr uint TP = 16u * P;
    constexpr int D = MT_DEPTH;
    const uint e = IDX ? found.e : blockIdx.y;
    const uint a0 = IDX ? 0u : min(offsets[e], NA), a1 = IDX ? found.n : min(offsets[e + 1], NA);
    if (a0 >= a1) return;
    const uint tid = threadIdx.x, lane = tid & 63u, nt = blockDim.x;
    const uint wave = (uint)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), nw = nt >> 6;
    const uint nsb = K >> 8, S = K + 16u, per_row = K >> 4;     // (rows 16 bytes past a bank period: 16 lanes' reads of 16 bytes cover every bank once)
    const uint o_lsx = TP * S, o_lbq = o_lsx + nsb * TP * 4u, o_zero = o_lbq + nsb * TP * 16u, o_av = o_zero + 256u;
    float* lsx = (float*)(lds + o_lsx);            // [sb][TP] token scales
    uchar* lbq = lds + o_lbq;                      // [sb][TP][16]: lo_0..7, hi_0..7 of the bsums
    uint* lav = (uint*)(lds + o_av);               // [TP] the pass's assignments
    const ushort* const lst = (const ushort*)(lds + MT_LDS - MT_LIST(found.n));    // (IDX: the expert's)
    if (tid < 64u) ((uint*)(lds + o_zero))[tid] = 0u;
    const uint n = lane & 15u, kg = lane >> 4;
    const size_t rb = (size_t)nsb * MtBytes<W>::N;
    const uint tiles = (N + 15u) >> 4;
    // copies of a unit: nine lanes per row, seven rows per copy (rows 14 and 15 in the third)
    const uint cq = lane / 9u, cpc16 = (lane - cq * 9u) * 16u, c_off = cq * (uint)rb + cpc16;
    // tile r of wave group g: (r groups + g) gridDim.x + blockIdx.x; a group is a wave, or a pair (even: gate, odd: up)
    const uint groups = GU ? nw >> 1 : nw, group = GU ? wave >> 1 : wave, stride = groups * gridDim.x;
    const uint first = group * gridDim.x + blockIdx.x, rounds = (tiles + stride - 1u) / stride;
    const uint my_tiles = first < tiles ? (tiles - first + stride - 1u) / stride : 0u;
    const uchar* const w = GU && (wave & 1u) ? w1 : w0;
    uchar* const own = lds + MT_LDS + wave * MtRing<W>::WAVE;
    const uint ring = (uint)(size_t)(__attribute__((address_space(3))) uchar*)lds + MT_LDS + wave * MtRing<W>::WAVE;
    const uchar* const rd = own + n * Q4K_BYTES;
    // the pieces of a unit that go through registers (past the last they repeat it)
    constexpr uint PC = DMA ? 1u : MtRing<W>::WAVE / 256u, NQ = (16u * PC + 63u) / 64u;
    typedef gq_i4 __attribute__((aligned(2))) piece;
    gq_i4 wv[NQ];
    uint wd = 0u;
    for (uint tt = a0; tt < a1; tt += TP) {
        const uint cnt = min(TP, a1 - tt);
        // This wave's tiles as one stream of units (16 rows at one super-block), copied by the memory system into the wave's
        // ring of D and asked for D units ahead across tile borders; the first D are on their way while the tokens are staged.
        const uint units = my_tiles * nsb;
        uint i_u = 0u, i_sb = 0u, i_tile = first, i_slot = 0u;
        auto issue_next = [&]() {
            const size_t at = (size_t)w + ((size_t)e * N + i_tile * 16u) * rb + (size_t)i_sb * MtBytes<W>::N;
            const uchar* base = (const uchar*)(((size_t)(uint)__builtin_amdgcn_readfirstlane((int)(at >> 32)) << 32) |
                                               (uint)__builtin_amdgcn_readfirstlane((int)(uint)at));   // (the copy wants it in scalar registers)
            if constexpr (DMA) {
                const uint dst = ring + i_slot * MT_UNIT;
                uint o0 = c_off, o1 = c_off + 7u * (uint)rb, o2 = c_off + 14u * (uint)rb;
                if (N - i_tile * 16u < 16u) {                          // the last tile of a ragged matrix: no row past N
                    const uint top = N - i_tile * 16u - 1u;
                    o0 = min(cq, top) * (uint)rb + cpc16;
                    o1 = min(7u + cq, top) * (uint)rb + cpc16;
                    o2 = min(14u + cq, top) * (uint)rb + cpc16;
                }
                if (lane < 63u) {
                    lds_dma16(base, o0, dst);
                    lds_dma16(base, o1, dst + 1008u);
                }
                if (lane < 18u) lds_dma16(base, o2, dst + 2016u);
                i_slot = i_slot + 1u == (uint)D ? 0u : i_slot + 1u;
            } else {
                const uint top = min(15u, N - i_tile * 16u - 1u);
#pragma unroll
                for (uint q = 0; q < NQ; q++) {
                    const uint p = min(lane + 64u * q, 16u * PC - 1u), r = p / PC;
                    wv[q] = *(const piece*)(base + (min(r, top) * (uint)rb + (p - r * PC) * 16u));
                }
                wd = W::tail(base + min(n, top) * (uint)rb);
            }
            i_u++;
            if (++i_sb == nsb) {
                i_sb = 0u;
                i_tile += stride;
            }
        };
        for (uint k = 0; k < (DMA ? (uint)D : 1u); k++)
            if (i_u < units) issue_next();
        __syncthreads();                           // the previous pass is done with the staged tokens
        if (!IDX && tid < TP) lav[tid] = min(list[min(tt + tid, a1 - 1u)], NA - 1u);
        auto assignment = [&](uint t) -> uint { return IDX ? lst[tt + t] : lav[t]; };      // the pass's t-th, t < cnt
        auto source = [&](uint t) {
            const uint av = IDX ? lst[tt + t] : min(list[min(tt + t, a1 - 1u)], NA - 1u);
            return GU ? av / KSEL : av;
        };
        if constexpr (QUANT) {
            // 32 lanes a segment of 256, eight values each, two segments' loads in flight: the operations of quantize_q8k
            const float* const act = (const float*)xq;
            const uint segs = cnt * nsb, l8 = (tid & 31u) * 8u;
            for (uint s0 = tid >> 5; s0 < segs; s0 += nt >> 4) {
                float4 v[2][2];
                uint t[2], sb[2];
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    const uint i = min(s0 + (uint)q * (nt >> 5), segs - 1u);
                    t[q] = i / nsb, sb[q] = i - t[q] * nsb;
                    const float4* const p = (const float4*)(act + (size_t)assignment(t[q]) * K + sb[q] * 256u + l8);
                    v[q][0] = p[0], v[q][1] = p[1];
                }
#pragma unroll
                for (int q = 0; q < 2; q++) {
                    float scale;
                    const uint2 c = oct_quant_q8k(v[q][0], v[q][1], scale);
                    int bs = dot4_i8(c.y, 0x01010101u, dot4_i8(c.x, 0x01010101u, 0));
                    bs += dpp_i32<OJK_DPP_QUAD_XOR1>(bs);
                    bs += dpp_i32<OJK_DPP_QUAD_XOR2>(bs);
                    if (s0 + (uint)q * (nt >> 5) < segs) {
                        uchar* const x = lds + (size_t)t[q] * S + sb[q] * 256u;
                        if constexpr (DMA) *(uint2*)(x + (l8 & ~63u) + ((l8 & 31u) << 1) + ((l8 & 32u) >> 2)) = c;
                        else *(uint2*)(x + l8) = c;
                        if ((tid & 3u) == 0u) {
                            lbq[(sb[q] * TP + t[q]) * 16u + (l8 >> 5)] = (uchar)(bs & 63);
                            lbq[(sb[q] * TP + t[q]) * 16u + 8u + (l8 >> 5)] = (uchar)(bs >> 6);
                        }
                        if (l8 == 0u) lsx[sb[q] * TP + t[q]] = scale;
                    }
                }
            }
            for (uint i = tid; i < nsb * (TP - cnt); i += nt) lsx[(i / (TP - cnt)) * TP + cnt + i % (TP - cnt)] = 0.0f;
            __syncthreads();
        } else {
            // token rows 0 .. cnt - 1, four loads of 16 bytes in flight per thread; two neighbours hold one run of 32 positions
            // and leave its sum (the even one the low part, the odd one the high part)
            const uint total = cnt * per_row;
            for (uint i0 = tid; i0 < total; i0 += 4u * nt) {
                uint4 v[4];
    #pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint i = min(i0 + (uint)q * nt, total - 2u + (tid & 1u)), t = i / per_row;
                    v[q] = *(const uint4*)(xq + (size_t)source(t) * K + ((i - t * per_row) << 4));
                }
    #pragma unroll
                for (int q = 0; q < 4; q++) {
                    const uint i = i0 + (uint)q * nt, t = i / per_row, o = (i - t * per_row) << 4;
                    int bs = dot4_i8(v[q].x, 0x01010101u, 0);
                    bs = dot4_i8(v[q].y, 0x01010101u, bs); bs = dot4_i8(v[q].z, 0x01010101u, bs); bs = dot4_i8(v[q].w, 0x01010101u, bs);
                    bs += dpp_i32<OJK_DPP_QUAD_XOR1>(bs);
                    if (i < total) {
                        if constexpr (DMA) {
                            uchar* const x = lds + (size_t)t * S + (o & ~63u) + ((o & 16u) << 1) + ((o & 32u) >> 2);
                            *(uint2*)x = make_uint2(v[q].x, v[q].y);
                            *(uint2*)(x + 16u) = make_uint2(v[q].z, v[q].w);
                        } else {
                            *(uint4*)(lds + (size_t)t * S + o) = v[q];
                        }
                        lbq[((o >> 8) * TP + t) * 16u + 8u * (tid & 1u) + ((o >> 5) & 7u)] = (uchar)((tid & 1u) ? bs >> 6 : bs & 63);
                    }
                }
            }
            for (uint i = tid; i < nsb * TP; i += nt) {
                const uint t = i / nsb, sb = i - t * nsb;
                lsx[sb * TP + t] = t < cnt ? xs[(size_t)source(t) * nsb + sb] : 0.0f;
            }
            __syncthreads();
        }
        const uint np = (cnt + 15u) >> 4;          // token tiles of 16 this pass holds
        const uchar* xa[P];
        uint xstep[P];
#pragma unroll
        for (int p = 0; p < P; p++) {
            const bool on = n + 16u * p < cnt;
            uint at = 16u * kg;
            if constexpr (!DMA) at = W::token_at(kg);
            xa[p] = on ? lds + (size_t)(n + 16u * p) * S + at : lds + o_zero + at;
            xstep[p] = on ? 256u : 0u;
        }
        uint c_tile = first, c_slot = 0u, u = 0u;
        for (uint r = 0; r < rounds; r++, c_tile += stride) {
            float acc[P][4];
#pragma unroll
            for (int p = 0; p < P; p++)
#pragma unroll
                for (int v = 0; v < 4; v++) acc[p][v] = 0.0f;
            const bool has = c_tile < tiles;
            if (has)
                for (uint sb = 0; sb < nsb; sb++, u++) {
                    if constexpr (DMA) {
                        if (units - u >= (uint)D) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(3 * (D - 1)) : "memory");
                        else asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
                        const uchar* blk = rd + c_slot * MT_UNIT;
                        c_slot = c_slot + 1u == (uint)D ? 0u : c_slot + 1u;
                        GqW c;
                        c.hdr = *(const uint4*)blk;
    #pragma unroll
                        for (int q = 0; q < 4; q++) c.q[q] = *(const uint2*)(blk + 16u + 32u * q + 8u * kg);
                        gq_i4 BA[4], BB[4];
                        const float d = f16_bits_to_f32(c.hdr.x & 0xFFFFu), dmin = f16_bits_to_f32(c.hdr.x >> 16);
                        const uint mn_lo = c.hdr.z & 0x3F3F3F3Fu;
                        const uint mn_hi = ((c.hdr.w >> 4) & 0x0F0F0F0Fu) | ((c.hdr.z >> 2) & 0x30303030u);
                        const long Bm = kg == 0u ? gq_pack(mn_lo, mn_hi) : 0;
                        gq_planes(c, BA, BB);
                        // the unit is in registers: its slot takes the unit D ahead
                        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                        if (i_u < units) issue_next();
                        __builtin_amdgcn_sched_barrier(0);
    #pragma unroll
                        for (int p = 0; p < P; p++)
                            if ((uint)p < np)
                                gq_planes_pass(BA, BB, Bm, d, dmin, xa[p] + sb * xstep[p], lbq + ((size_t)sb * TP + 16u * p + n) * 16u,
                                               lsx + sb * TP + 16u * p, kg, acc[p]);
                    } else {
#pragma unroll
                        for (uint q = 0; q < NQ; q++) *(gq_i4*)(own + min(lane + 64u * q, 16u * PC - 1u) * 16u) = wv[q];
                        if (16u * PC < MtBytes<W>::N) ((ushort*)(own + 256u * PC))[n] = (ushort)wd;
                        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                        __builtin_amdgcn_wave_barrier();
                        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                        W c;
                        c.read(own + n * (16u * PC), kg, ((const ushort*)(own + 256u * PC))[n]);
                        if (i_u < units) issue_next();
                        gq_i4 BH[4], BL[4];
                        c.planes(kg, BH, BL);
                        const float dh = 0.5f * c.d(), dmin = c.dmin();      // (the digits are of twice the integers)
                        const long Bm = c.mins(kg);
#pragma unroll
                        for (int p = 0; p < P; p++)
                            if ((uint)p < np)
                                mt_digits_pass<W>(BH, BL, Bm, dh, dmin, xa[p] + sb * xstep[p], lbq + ((size_t)sb * TP + 16u * p + n) * 16u,
                                                  lsx + sb * TP + 16u * p, kg, acc[p]);
                    }
                }
            // D register v of lane (n, kg): assignment 16 p + 4 kg + v of the pass, row n of the tile
            const bool mine = has && c_tile * 16u + n < N;
#pragma unroll
            for (int p = 0; p < P; p++) {
                if ((uint)p >= np) break;
                float* const ex = (float*)(lds + MT_LDS + MT_RING) + ((wave >> 1) * 64u + lane) * 4u;
                float up[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                if (GU) {
                    if (wave & 1u) *(float4*)ex = make_float4(acc[p][0], acc[p][1], acc[p][2], acc[p][3]);
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                    if ((wave & 1u) == 0u) {
                        const float4 t = *(const float4*)ex;
                        up[0] = t.x, up[1] = t.y, up[2] = t.z, up[3] = t.w;
                    }
                    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
                    __builtin_amdgcn_s_barrier();
                }
                if (mine && (!GU || (wave & 1u) == 0u)) {
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const uint t = 16u * p + 4u * kg + (uint)v;
                        if (t < cnt) {
                            const float g = acc[p][v];
                            out[(size_t)assignment(t) * N + c_tile * 16u + n] = GU ? (g / (1.0f + expf(-g))) * up[v] : g;
                        }
                    }
                }
            }
        }
    }
}

#define MT_FITS(P, LIST) (16u * P * (K + 32u) + 5u * P * (K >> 2) + (LIST) + 256u <= MT_LDS)
#define MT_PICK(W, GU, IDX, COUNT, X, S, W0, W1, OUT, KS)                                                              \
    do {                                                                                                              \
        if (COUNT > 48u && MT_FITS(4u, IDX ? MT_LIST(COUNT) : 64u * 4u)) moe_mt_body<W, GU, IDX, 4>(X, S, W0, W1, OUT, offsets, list, K, N, KS, NA, lds_mt, found); \
        else if (COUNT > 32u && MT_FITS(3u, IDX ? MT_LIST(COUNT) : 64u * 3u)) moe_mt_body<W, GU, IDX, 3>(X, S, W0, W1, OUT, offsets, list, K, N, KS, NA, lds_mt, found); \
        else if (COUNT > 16u && MT_FITS(2u, IDX ? MT_LIST(COUNT) : 64u * 2u)) moe_mt_body<W, GU, IDX, 2>(X, S, W0, W1, OUT, offsets, list, K, N, KS, NA, lds_mt, found); \
        else moe_mt_body<W, GU, IDX, 1>(X, S, W0, W1, OUT, offsets, list, K, N, KS, NA, lds_mt, found);                \
    } while (0)
#define MT_RUN(W, GU, X, S, W0, W1, OUT, KS)                                                                           \
    const MtFound found = {};                                                                                         \
    const uint n_ = min(offsets[blockIdx.y + 1u], NA) - min(offsets[blockIdx.y], NA);                                 \
    MT_PICK(W, GU, false, n_, X, S, W0, W1, OUT, KS)
#define MT_RUN_IDX(W, GU, X, S, W0, W1, OUT, KS)                                                                       \
    const uint *const offsets = nullptr, *const list = nullptr;                                                       \
    const MtFound found = mt_find(idx, NA, E, lds_mt);                                                                \
    MT_PICK(W, GU, true, found.n, X, S, W0, W1, OUT, KS)
extern "C" __global__ void __launch_bounds__(1024)
moe_gu_q4k_mt(const signed char* __restrict__ xq, const float* __restrict__ xs, const uchar* __restrict__ wg,
              const uchar* __restrict__ wu, float* __restrict__ act, const uint* __restrict__ offsets,
              const uint* __restrict__ list, uint K, uint N, uint KSEL, uint NA) {
    __shared__ __attribute__((aligned(16))) uchar lds_mt[MT_LDS + MT_RING + 8192u];
    MT_RUN(MtQ4K, true, xq, xs, wg, wu, act, KSEL);
}
//   moe_gu_q4k_ti(xq, xs, wg, wu, act, idx, K, N, KSEL, NA, E)   moe_down_{q4k,q5k,q6k}_ti(act, wd, dv, idx, K, N, NA, E)
//                                                                grid [1 .. ceil(N / 16), min(E, NA), 1], block 512 or 1024
// the same over at most 4096 assignments as the router leaves them: a workgroup finds its expert's among idx itself (two or
// eight loads a thread), and the down entries quantize the f32 activations while they stage them.  The grouping's and the
// quantizer's launches are gone, 3 us of dispatch each: 128 experts of 768 x 2048, the
// layer at 256 tokens 108.0 -> 103.9 us, at 64 92.6 -> 88.6; 32 of 512 x 1024 at 12 31.3 -> 23.8.
extern "C" __global__ void __launch_bounds__(1024)
moe_gu_q4k_ti(const signed char* __restrict__ xq, const float* __restrict__ xs, const uchar* __restrict__ wg,
              const uchar* __restrict__ wu, float* __restrict__ act, const uint* __restrict__ idx, uint K, uint N, uint KSEL, uint NA, uint E) {
    __shared__ __attribute__((aligned(16))) uchar lds_mt[MT_LDS + MT_RING + 8192u];
    MT_RUN_IDX(MtQ4K, true, xq, xs, wg, wu, act, KSEL);
}

#define MOE_DOWN_MT(FMT, W)                                                                                            \
    extern "C" __global__ void __launch_bounds__(1024)                                                                \
    moe_down_##FMT##_mt(const signed char* __restrict__ aq, const float* __restrict__ as_, const uchar* __restrict__ wd, \
                        float* __restrict__ dv, const uint* __restrict__ offsets, const uint* __restrict__ list,       \
                        uint K, uint N, uint NA) {                                                                     \
        __shared__ __attribute__((aligned(16))) uchar lds_mt[MT_LDS + 16u * MtRing<W>::WAVE];                          \
        MT_RUN(W, false, aq, as_, wd, wd, dv, 1u);                                                                     \
    }                                                                                                                  \
    extern "C" __global__ void __launch_bounds__(1024)                                                                \
    moe_down_##FMT##_ti(const float* __restrict__ act, const uchar* __restrict__ wd, float* __restrict__ dv,           \
                        const uint* __restrict__ idx, uint K, uint N, uint NA, uint E) {                               \
        __shared__ __attribute__((aligned(16))) uchar lds_mt[MT_LDS + 16u * MtRing<W>::WAVE];                          \
        MT_RUN_IDX(W, false, (const signed char*)act, nullptr, wd, wd, dv, 1u);                                        \
    }
MOE_DOWN_MT(q4k, MtQ4K)
MOE_DOWN_MT(q5k, MtQ5K)
MOE_DOWN_MT(q6k, MtQ6K)
#undef MT_PICK
#undef MT_RUN_IDX
#undef MT_RUN

// ------------------------------------------------------------------ combine
// y[t][i] (=, +=) sum_j wgt[t][j] * dv[t*KSEL + j][i], slots in order.
extern "C" __global__ void __launch_bounds__(256)
moe_combine(const float* __restrict__ dv, const float* __restrict__ wgt, float* __restrict__ y,
            uint T, uint KSEL, uint D, uint ACC) {
    const size_t i = (size_t)blockIdx.x * 256u + threadIdx.x;
    if (i >= (size_t)T * D) return;
    const uint t = (uint)(i / D), col = (uint)(i % D);
    float acc = ACC ? y[i] : 0.0f;
    // (eight slots' loads in flight before the first is added — slot order kept; past the last slot they repeat it)
    for (uint j0 = 0; j0 < KSEL; j0 += 8u) {
        float w[8], d[8];
#pragma unroll
        for (int u = 0; u < 8; u++) {
            const size_t a = (size_t)t * KSEL + min(j0 + (uint)u, KSEL - 1u);
            w[u] = wgt[a];
            d[u] = dv[a * D + col];
        }
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (j0 + (uint)u < KSEL) acc += w[u] * d[u];
    }
    y[i] = acc;
}

// ------------------------------------------------------------------ K-quant experts on f32 activations
// The reference's expert kernels for raw K-quant rows under their own names (the expert table,
// crates/ojas-core/src/quant_src.rs:168-193; bodies crates/ojas-metal/src/kernels/moe.rs:497-527, :722-815), with
// the argument lists of the Q8_0 pair above:
//   moe_gu_q4k(x, wg, wu, act, idx, K, N)              moe_down_{q5k,q6k}(act, wd, y, idx, wgt, K, N, KSEL)
// f32 activations meet the dequantized weights (the float contract; the CPU path's int8-activation arithmetic is
// what the _dec / _m / _mm / _mt entries above compute).  moe_down_q4k is this library's addition, so that an
// all-Q4_K layer runs under the same contract.
MOE_ROWS_GU_ENTRY(q4k, Q4kW)
MOE_ROWS_DOWN_ENTRY(q4k, Q4kW)
MOE_ROWS_DOWN_ENTRY(q5k, Q5kW)
MOE_ROWS_DOWN_ENTRY(q6k, Q6kW)
