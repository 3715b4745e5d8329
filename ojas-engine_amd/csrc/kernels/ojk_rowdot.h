// Matvec bodies driven by a row trait (ojk_rows.h, ojk_iq_grid_rows.h): raw rows of a block format against f32
// activations, shared by the code objects that hold such formats.  A trait W gives the lane map of one wave step
// and load / dot for the lane's fragment of a block.
#pragma once
#include "ojk_common.h"

enum { ST_SET = 0, ST_ACCUM = 1, ST_BIAS = 2 };

template <int MODE>
__device__ __forceinline__ void store_row(float* y, const float* bs, uint n, float v) {
    if (MODE == ST_SET) y[n] = v;
    else if (MODE == ST_ACCUM) y[n] += v;
    else y[n] = v + bs[n];
}

template <class W, int R, int MODE>
__device__ __forceinline__ void gemv_nat_iq4_body(const float* __restrict__ x, const uchar* __restrict__ w,
                                                  float* __restrict__ y, const float* __restrict__ bs,
                                                  uint K, uint N) {
    const uint lane = threadIdx.x & 63u;
    const uint row0 = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * R;
    if (row0 >= N) return;
    const uint nu = W::units(K);
    const size_t rb = (size_t)nu * W::BYTES;
    float acc[R];
#pragma unroll
    for (int r = 0; r < R; r++) acc[r] = 0.0f;
    for (uint u = W::unit_of(lane); u < nu; u += W::STEP) {
        typename W::Frag f[R];
#pragma unroll
        for (int r = 0; r < R; r++) f[r] = W::load(w + (size_t)min(row0 + r, N - 1u) * rb, u, lane);
        const float* xp = x + (size_t)u * W::x_unit(0) + W::x_off(lane);
        const float4 x0 = *(const float4*)xp, x1 = *(const float4*)(xp + W::XGAP);
        const float xsum = sum4(x0) + sum4(x1);      // for the formats with an offset or a minimum
#pragma unroll
        for (int r = 0; r < R; r++) acc[r] += W::dot(f[r], lane, x0, x1, xsum);
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
        float s = wave_sum(acc[r]);
        if (lane == 0 && row0 + r < N) store_row<MODE>(y, bs, row0 + r, s);
    }
}

template <class W, int MT>
__device__ __forceinline__ void gemv_nat_iq4_m_body(const float* __restrict__ x, const uchar* __restrict__ w,
                                                    float* __restrict__ y, uint K, uint N, uint M, uint ACC) {
    const uint lane = threadIdx.x & 63u;
    const uint row = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    if (row >= N) return;
    const uint nu = W::units(K);
    const uchar* wr = w + (size_t)row * nu * W::BYTES;
    for (uint m0 = 0; m0 < M; m0 += MT) {
        float acc[MT];
#pragma unroll
        for (int i = 0; i < MT; i++) acc[i] = 0.0f;
        for (uint u = W::unit_of(lane); u < nu; u += W::STEP) {
            const typename W::Frag f = W::load(wr, u, lane);
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const uint m = min(m0 + i, M - 1u);
                const float* xp = x + (size_t)m * K + (size_t)u * W::x_unit(0) + W::x_off(lane);
                const float4 x0 = *(const float4*)xp, x1 = *(const float4*)(xp + W::XGAP);
                acc[i] += W::dot(f, lane, x0, x1, sum4(x0) + sum4(x1));
            }
        }
#pragma unroll
        for (int i = 0; i < MT; i++) {
            float s = wave_sum(acc[i]);
            if (lane == 0 && m0 + i < M) {
                float* o = y + (size_t)(m0 + i) * N + row;
                *o = ACC ? *o + s : s;
            }
        }
    }
}

// Two tokens and more against many steps of K: gemv_nat_<fmt>_ms(x, w, y, K, N, M, ACC), the _m entry's arguments and grid.  A workgroup of
// n waves owns n rows, four at a time; its waves take a step of K each in turn for all four rows, and their sums meet in LDS
// in wave order.  A lane's f32 activations, 8 bytes a weight at two tokens, are what such a call asks the address unit for: a wave
// that walks a row by itself fetches them again for every row.  Whole call, _m / _ms, us: IQ4_XS 14336 x 4096 at 3 tokens 37.4 / 17.7,
// 4096 x 14336 at 2 19.8 / 15.0, 27347 x 13312 at 3 259 / 94.6; Q8_0 14336 x 4096 at 2 22.5 / 15.2, at 3 35.5 / 17.2.  With few steps of K
// some waves have none: 30000 x 1280 IQ4_XS at 2 16.2 / 18.1, at 3 28.8 / 20.4, 1599 x 1024 at 4 4.4 / 4.7 (two waves on two rows there: 21.9 and 24.6).
// More than four tokens (f32 activations asked for, a K without a tile) are further passes of four over the rows, as in the _m entry:
// Q8_0 4096 x 4096 at 5 24.0 / 16.4, at 16 41.5 / 27.8, at 31 76.5 / 48.8, 14336 x 1280 at 9 42.2 / 30.7, 4096 x 14336 at 31 268 / 176; Q5_0
// 1001 x 2304 at 8 13.0 / 8.9, IQ4_XS 2000 x 1280 at 64 42.2 / 38.5, 4096 x 4096 at 300 801 / 398: ahead at each of 8 shapes.
template <class W, int MT>
__device__ __forceinline__ void gemv_nat_ms_body(const float* __restrict__ x, const uchar* __restrict__ w,
                                                 float* __restrict__ y, uint K, uint N, uint M, uint ACC) {
    constexpr uint R = 4u;
    __shared__ float red[16][MT][R];
    const uint lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const uint nu = W::units(K), first = blockIdx.x * nw, end = min(first + nw, N);
    const size_t rb = (size_t)nu * W::BYTES;
    for (uint row0 = first; row0 < end; row0 += R) {
        for (uint m0 = 0; m0 < M; m0 += MT) {
            float acc[MT][R];
#pragma unroll
            for (int i = 0; i < MT; i++)
#pragma unroll
                for (uint r = 0; r < R; r++) acc[i][r] = 0.0f;
            for (uint u = W::unit_of(lane) + wave * W::STEP; u < nu; u += nw * W::STEP) {
                typename W::Frag f[R];
#pragma unroll
                for (uint r = 0; r < R; r++) f[r] = W::load(w + (size_t)min(row0 + r, end - 1u) * rb, u, lane);
#pragma unroll
                for (int i = 0; i < MT; i++) {
                    const float* xp = x + (size_t)min(m0 + i, M - 1u) * K + (size_t)u * W::x_unit(0) + W::x_off(lane);
                    const float4 x0 = *(const float4*)xp, x1 = *(const float4*)(xp + W::XGAP);
                    const float xsum = sum4(x0) + sum4(x1);
#pragma unroll
                    for (uint r = 0; r < R; r++) acc[i][r] += W::dot(f[r], lane, x0, x1, xsum);
                }
            }
            if (row0 > first || m0 > 0u) __syncthreads();       // the sums before have been read
#pragma unroll
            for (int i = 0; i < MT; i++) {
                const float t = wave_sum4(acc[i][0], acc[i][1], acc[i][2], acc[i][3], lane);
                if (lane < R) red[wave][i][lane] = t;
            }
            __syncthreads();
            const uint i = threadIdx.x / R, r = threadIdx.x % R;
            if (i < (uint)MT && m0 + i < M && row0 + r < end) {
                float t = red[0][i][r];
                for (uint v = 1; v < nw; v++) t += red[v][i][r];
                float* o = y + (size_t)(m0 + i) * N + row0 + r;
                *o = ACC ? *o + t : t;
            }
        }
    }
}
#define GEMV_NAT_MS(FMT, W)                                                                                \
    extern "C" __global__ void __launch_bounds__(256) gemv_nat_##FMT##_ms(                                 \
        const float* x, const uchar* w, float* y, uint K, uint N, uint M, uint ACC) {                      \
        if (M <= 2) gemv_nat_ms_body<W, 2>(x, w, y, K, N, M, ACC);                                         \
        else if (M == 3) gemv_nat_ms_body<W, 3>(x, w, y, K, N, M, ACC);                                    \
        else gemv_nat_ms_body<W, 4>(x, w, y, K, N, M, ACC); }

// Many rows (an output head): a 4-bit row is an eighth of the bytes of the f32 activations it meets, so
// a wave that fetches its activation fragments again for every few rows is bound by those loads, not
// by HBM (2.7 TB/s at 128256 x 4096).  Here rows are grid-stride and the wave keeps its share of x —
// 8 floats per lane and step, NS steps — in registers for the whole launch; out-of-range steps hold
// zeros and repeat the last block.   gemv_nat_iq4{nl,xs}_px(x, w, y, K, N), K <= 4096 (64 floats of x per
// lane; twice that would halve the resident waves).
template <class W, int NS>
__device__ __forceinline__ void gemv_nat_iq4_px_body(const float* __restrict__ x, const uchar* __restrict__ w,
                                                     float* __restrict__ y, uint K, uint N) {
    const uint lane = threadIdx.x & 63u;
    const uint nu = W::units(K);
    const size_t rb = (size_t)nu * W::BYTES;
    float4 xr[NS][2];
    float xsum[NS];
    uint uc[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const uint u = W::unit_of(lane) + (uint)s * W::STEP;
        uc[s] = min(u, nu - 1u);
        xr[s][0] = xr[s][1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (u < nu) {
            const float* xp = x + (size_t)u * W::x_unit(0) + W::x_off(lane);
            xr[s][0] = *(const float4*)xp;
            xr[s][1] = *(const float4*)(xp + W::XGAP);
        }
        xsum[s] = sum4(xr[s][0]) + sum4(xr[s][1]);
    }
    const uint nwaves = gridDim.x * (blockDim.x >> 6);
    for (uint row0 = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 2u; row0 < N; row0 += nwaves * 2u) {
        const uchar* r0 = w + (size_t)row0 * rb;
        const uchar* r1 = w + (size_t)min(row0 + 1u, N - 1u) * rb;
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const typename W::Frag f0 = W::load(r0, uc[s], lane), f1 = W::load(r1, uc[s], lane);
            a0 += W::dot(f0, lane, xr[s][0], xr[s][1], xsum[s]);
            a1 += W::dot(f1, lane, xr[s][0], xr[s][1], xsum[s]);
        }
        a0 = wave_sum(a0);
        a1 = wave_sum(a1);
        if (lane == 0) {
            y[row0] = a0;
            if (row0 + 1u < N) y[row0 + 1u] = a1;
        }
    }
}

// The head form with a lane per 32-weight group: lane l of step s owns group l + 64 s of the row (its 16 code bytes in
// one load where the group-per-four-lanes map above issues four narrow ones — the address unit of the vector memory
// path takes a wave-wide load about as long whatever its width, and bounds those launches) and keeps the group's 32
// activations, and their sum, in registers.  A trait T gives row_bytes(K) and dot32(row, group, x[8], xsum): the
// group's term with its scale.  K <= 4096 (two steps).
template <class T>
__device__ __forceinline__ void gemv_nat_sub32_px_body(const float* __restrict__ x, const uchar* __restrict__ w,
                                                       float* __restrict__ y, uint K, uint N) {
    constexpr int NS = 2;
    const uint lane = threadIdx.x & 63u, nsub = K >> 5;
    const size_t rb = T::row_bytes(K);
    float4 xr[NS][8];
    float xsum[NS];
    uint sc[NS];
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const uint sub = lane + 64u * (uint)s;
        sc[s] = min(sub, nsub - 1u);
        float t = 0.0f;
#pragma unroll
        for (int j = 0; j < 8; j++) {
            xr[s][j] = sub < nsub ? *(const float4*)(x + (size_t)sub * 32u + 4u * (uint)j) : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            t += (xr[s][j].x + xr[s][j].y) + (xr[s][j].z + xr[s][j].w);
        }
        xsum[s] = t;
    }
    const uint nwaves = gridDim.x * (blockDim.x >> 6);
    for (uint row0 = (blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6)) * 2u; row0 < N; row0 += nwaves * 2u) {
        const uchar* r0 = w + (size_t)row0 * rb;
        const uchar* r1 = w + (size_t)min(row0 + 1u, N - 1u) * rb;
        float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            a0 += T::dot32(r0, sc[s], xr[s], xsum[s]);
            a1 += T::dot32(r1, sc[s], xr[s], xsum[s]);
        }
        a0 = wave_sum(a0);
        a1 = wave_sum(a1);
        if (lane == 0) {
            y[row0] = a0;
            if (row0 + 1u < N) y[row0 + 1u] = a1;
        }
    }
}
#define GEMV_NAT_SUB32_PX(FMT, T)                                                                          \
    extern "C" __global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(4, 4)))           \
    gemv_nat_##FMT##_px(const float* x, const uchar* w, float* y, uint K, uint N) {                        \
        gemv_nat_sub32_px_body<T>(x, w, y, K, N); }

#define GEMV_NAT_IQ4_PX(FMT, W)                                                                            \
    extern "C" __global__ void __launch_bounds__(256) gemv_nat_##FMT##_px(                                 \
        const float* x, const uchar* w, float* y, uint K, uint N) {                                        \
        gemv_nat_iq4_px_body<W, 8>(x, w, y, K, N); }

// The reference's entry set of one format: gemv_nat_<fmt>{,_r1,_r2,_accum,_bias,_m}, over gemv_nat_<fmt>_body<R, MODE>
// and gemv_nat_<fmt>_m_body<MT>.
#define GEMV_NAT_ENTRIES(FMT)                                                                              \
    extern "C" __global__ void __launch_bounds__(256) gemv_nat_##FMT##_r1(                                 \
        const float* x, const uchar* w, float* y, uint K, uint N) {                                        \
        gemv_nat_##FMT##_body<1, ST_SET>(x, w, y, nullptr, K, N); }                                        \
    extern "C" __global__ void __launch_bounds__(256) gemv_nat_##FMT##_r2(                                 \
        const float* x, const uchar* w, float* y, uint K, uint N) {                                        \
        gemv_nat_##FMT##_body<2, ST_SET>(x, w, y, nullptr, K, N); }                                        \
    extern "C" __global__ void __launch_bounds__(256) gemv_nat_##FMT(                                      \
        const float* x, const uchar* w, float* y, uint K, uint N) {                                        \
        gemv_nat_##FMT##_body<4, ST_SET>(x, w, y, nullptr, K, N); }                                        \
    extern "C" __global__ void __launch_bounds__(256) gemv_nat_##FMT##_accum(                              \
        const float* x, const uchar* w, float* y, uint K, uint N) {                                        \
        gemv_nat_##FMT##_body<4, ST_ACCUM>(x, w, y, nullptr, K, N); }                                      \
    extern "C" __global__ void __launch_bounds__(256) gemv_nat_##FMT##_bias(                               \
        const float* x, const uchar* w, float* y, const float* bs, uint K, uint N) {                       \
        gemv_nat_##FMT##_body<4, ST_BIAS>(x, w, y, bs, K, N); }                                            \
    extern "C" __global__ void __launch_bounds__(256) gemv_nat_##FMT##_m(                                  \
        const float* x, const uchar* w, float* y, uint K, uint N, uint M, uint ACC) {                      \
        if (M <= 2) gemv_nat_##FMT##_m_body<2>(x, w, y, K, N, M, ACC);                                     \
        else gemv_nat_##FMT##_m_body<4>(x, w, y, K, N, M, ACC); }

