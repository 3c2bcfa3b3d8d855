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

// The epilogue of a wave's four rows, an element to a lane (lanes 0 to 3; pairs: 0 and 1).  What it reads is requested ahead of the weights: at
// the end it is a round trip of its own, two where the position stands between (rotations), and one lane working all four elements takes four
// times as long over their exponentials.  The operations are dense_epilogue's.
template <typename T, DenseEpi MODE>
struct RowEpilogue {
    float pw = 0.f, pb = 0.f, nw = 0.f, nb = 0.f, x = 0.f;      // Residual: the norms' weights, the stream; Rope: cosine and sine in pw, pb
    T gate = (T)0.0f;
    uint32_t n0, i, pair = 0, pos = 0;
    bool rotates = false;

    __device__ __forceinline__ RowEpilogue(const DenseEpiArgs& e, uint32_t n0_, uint32_t N, uint32_t lane) : n0(n0_), i(lane & 3) {
        const uint32_t n = min(n0 + i, N - 1);
        if constexpr (MODE == DenseEpi::Residual) {
            if (e.post.w) { pw = e.post.w[n]; pb = e.post.b[n]; }
            if (e.next.w) { nw = e.next.w[n]; nb = e.next.b[n]; }
            if (e.add) x = e.f32[n];
        }
        if constexpr (MODE == DenseEpi::GateMul) gate = ((const T*)e.gate)[n];
        if constexpr (MODE == DenseEpi::Rope) {
            const uint32_t j = n0 % e.head_stride;
            pair = (j - e.rot_off) / 2 + (i >> 1);
            rotates = j >= e.rot_off && pair < e.rot_pairs;
            pos = e.pos_dev ? *e.pos_dev : e.base_pos;
        }
    }
    // behind the weights' requests: what an address had to be waited for
    __device__ __forceinline__ void late(const DenseEpiArgs& e) {
        if constexpr (MODE == DenseEpi::Rope) {
            if (rotates) { pw = e.cos_t[(size_t)pos * e.rot_pairs + pair]; pb = e.sin_t[(size_t)pos * e.rot_pairs + pair]; }
        }
    }
    __device__ __forceinline__ void store(const DenseEpiArgs& e, uint32_t N, uint32_t lane, const float (&v)[4]) const {
        if (lane >= 4) return;
        const uint32_t n = n0 + i;
        float a = i == 0 ? v[0] : i == 1 ? v[1] : i == 2 ? v[2] : v[3];
        if constexpr (MODE == DenseEpi::F32) {
            if (n < N) e.f32[n] = e.cap > 0.f ? e.cap * tanhf(a / e.cap) : a;
        } else if constexpr (MODE == DenseEpi::RawGate) {
            if (n0 < e.split) e.f32[n] = a;
            else ((T*)e.out)[n - e.split] = (T)act_f(e.act, a);
        } else if constexpr (MODE == DenseEpi::Rope) {
            const float b = i == 0 ? v[1] : i == 1 ? v[0] : i == 2 ? v[3] : v[2];
            if (rotates) a = i & 1 ? a * pw + b * pb : a * pw - b * pb;
            ((T*)e.out)[n] = (T)a;
        } else if constexpr (MODE == DenseEpi::GateMul) {
            ((T*)e.out)[n] = (T)(a * (float)gate);
        } else if constexpr (MODE == DenseEpi::ActPair) {
            if (i < 2) ((T*)e.out)[n0 / 2 + i] = (T)(act_f(e.act, i ? v[2] : v[0]) * (i ? v[3] : v[1]));
        } else {
            static_assert(MODE == DenseEpi::Residual, "the modes of a row");
            if (e.post.w) a = tanhf(e.post.alpha * a) * pw + pb;
            a += x;
            e.f32[n] = a;
            if (!e.out) return;
            if (e.next.w) a = tanhf(e.next.alpha * a) * nw + nb;
            ((T*)e.out)[n] = (T)a;
        }
    }
};

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
    RowEpilogue<T, MODE> epilogue(e, n0, N, lane);
    __builtin_amdgcn_sched_barrier(0);
    fetch(va, k_lane);
    if constexpr (STEPS > 1) fetch(vb, k_lane + D);
    __builtin_amdgcn_sched_barrier(0);
    epilogue.late(e);
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
    if (part == 0 && n0 < N) epilogue.store(e, N, lane, acc);
}

// Depth split of an N-row matrix: as many waves per row group as it takes to have a few workgroups on every compute unit.
inline int gemv_depth_split(uint32_t N, uint32_t K) {
    if (N / 16 >= 768 || K <= 512) return 1;
    if (N / 8 >= 768 || K <= 1024) return 2;
    return 4;
}

}  // namespace fh
