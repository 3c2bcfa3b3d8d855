// One row times a dense matrix: the body that the matrix-vector kernels share.  A wave works 4 consecutive matrix rows; KS waves
// split the depth of the same 4 rows (small matrices: enough loads in flight on every compute unit).
//
// What bounds it: the matrix is read once.  Two steps of weights (16 loads of 16 bytes per lane in bfloat16, all a wave has to read up
// to a depth of 2048 KS) are requested before the prologue prepares the vector in LDS, and from then on a step is requested as soon as
// its registers are free.  Loads come back in the order of their requests, so a kernel whose prologue reads global memory requests that
// ahead of the weights, into registers: behind them it would wait for all of them.  bfloat16, one step ahead and the vector last /
// this form: 16384 x 2048 16.2 / 14.9 us (4.5 TB/s with the launch), 2048 x 8192 10.2 / 9.5, 128256 x 2048 95.0 / 92.5.
// A depth that one step covers (STEPS = 1) has nothing to request ahead and leaves those instructions out: 576 x 576 2.9 / 2.7 us.
#pragma once

#include "dense.h"

namespace fh {

constexpr uint32_t GEMV_THREADS = 256;
template <int KS> constexpr uint32_t gemv_rows() { return 4 * (GEMV_THREADS / 64) / KS; }    // matrix rows of a workgroup

template <typename T> constexpr uint32_t gemv_unroll() { return sizeof(T) == 2 ? 2 : 1; }
// matrix columns that the waves of a row group work in one step
template <typename T, int KS> constexpr uint32_t gemv_step() { return gemv_unroll<T>() * KS * 512; }

// xs: LDS, K floats, filled by `prologue`; red: LDS, 16 floats.  STEPS = 1: K <= gemv_step.
template <typename T, int KS, DenseEpi MODE, int STEPS, typename Prologue>
__device__ __forceinline__ void gemv_body(const T* __restrict__ w, uint32_t N, uint32_t K, uint32_t row0, float* xs, float* red,
                                          const DenseEpiArgs& e, Prologue prologue) {
    typedef typename Vec<T>::x8 x8;
    constexpr int U = gemv_unroll<T>();
    constexpr uint32_t STEP = KS * 512;
    const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const uint32_t part = wave % KS, n0 = row0 + (wave / KS) * 4;
    const T* rows[4];
#pragma unroll
    for (int i = 0; i < 4; i++) rows[i] = w + (size_t)min(n0 + i, N - 1) * K;
    const uint32_t k_lane = (part * 64 + lane) * 8;
    auto fetch = [&](x8 (&v)[U][4], uint32_t k) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (k + u * STEP >= K) break;             // `add` stops there too
#pragma unroll
            for (int i = 0; i < 4; i++) v[u][i] = load8(rows[i] + k + u * STEP);
        }
    };
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    auto add = [&](const x8 (&v)[U][4], uint32_t k) {
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (k + u * STEP >= K) break;
            const v4f xa = *reinterpret_cast<const v4f*>(xs + k + u * STEP), xb = *reinterpret_cast<const v4f*>(xs + k + u * STEP + 4);
#pragma unroll
            for (int i = 0; i < 4; i++) {
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i] = fmaf((float)v[u][i][j], xa[j], acc[i]);
#pragma unroll
                for (int j = 0; j < 4; j++) acc[i] = fmaf((float)v[u][i][4 + j], xb[j], acc[i]);
            }
        }
    };
    x8 va[U][4], vb[U][4];
    constexpr uint32_t D = U * STEP;
    __builtin_amdgcn_sched_barrier(0);
    fetch(va, k_lane);
    if constexpr (STEPS > 1) fetch(vb, k_lane + D);
    __builtin_amdgcn_sched_barrier(0);
    prologue();
    __syncthreads();
    if constexpr (STEPS == 1) add(va, k_lane);
    else {
        for (uint32_t k = 0; k < K; k += 2 * D) {
            add(va, k_lane + k);
            if (k + 2 * D < K) fetch(va, k_lane + k + 2 * D);
            add(vb, k_lane + k + D);
            if (k + 3 * D < K) fetch(vb, k_lane + k + 3 * D);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; i++) acc[i] = wave_sum(acc[i]);
    if (KS > 1) {
        if (lane == 0) {
#pragma unroll
            for (int i = 0; i < 4; i++) red[wave * 4 + i] = acc[i];
        }
        __syncthreads();
#pragma unroll
        for (int p = 1; p < KS; p++)
#pragma unroll
            for (int i = 0; i < 4; i++)
                if (part == 0) acc[i] += red[(wave + p) * 4 + i];
    }
    if (part == 0 && lane == 0 && n0 < N) dense_epilogue<T, MODE>(e, 0, n0, N, acc, epilogue_cols<MODE>(e, n0), epilogue_row<T, MODE>(e, 0, n0));
}

// Depth split of an N-row matrix: as many waves per row group as it takes to have a few workgroups on every compute unit.
inline int gemv_depth_split(uint32_t N, uint32_t K) {
    if (N / 16 >= 768 || K <= 512) return 1;
    if (N / 8 >= 768 || K <= 1024) return 2;
    return 4;
}

}  // namespace fh
