// Products with dense matrices (bfloat16 or 32-bit), y = a W^T, and the small kernels around them.
//
// M > 1: tiles on the matrix unit.  Workgroup = WN x WM x KG waves, each TN x TM tiles of 32 x 32 over a KG-th of every stage's depth;
// the weights are the MFMA A operand, so a lane ends up with four consecutive columns n of one row m (pairs of columns, rotary pairs
// and gate / up in one lane).  A stage of 128 bytes of depth (64 bfloat16, 32 floats) goes from global memory straight into one of NBUF
// LDS buffers while another one is worked; LDS rows are 128 bytes, the 16-byte piece c of row r at position c ^ ((r >> 1) & 7), which
// keeps the fragment reads free of bank conflicts.  Rows past the end of a matrix read as zero through the buffer descriptors' range
// check.
//
// What bounds it (bfloat16; matrix unit busy 31 % of 16384 x 2048 by 902 rows before, LDS 16 %, no bank conflicts):
// - The results.  A lane holds 16 bytes of a row and its neighbours other rows, so stores straight from the registers touched a cache
//   line per lane: 6 us for a tile of 128 x 128, 24 us for 256 x 256.  They go through LDS and out by whole rows.
// - Operands that several XCDs fetch.  Tiles are dealt out in groups of a few rows of tiles, column by column, and an XCD works a run of
//   them: at 902 rows each XCD reads a part of the weights where it used to read all of them.
// - The latency of a stage's loads where a compute unit has one workgroup: 3 or 4 buffers, and the depth shared out to the waves.
// Times in us of a caller's loop, 32-bit results, before / now: 16384 x 2048 by 902 rows 110 / 66.5 (910 TFLOP/s), 2048 x 8192 by 902
// 67.9 / 47.1, 2048 x 2048 by 902 22.9 / 15.3, 6144 x 2048 by 902 48.4 / 32.2, 3072 x 576 by 2502 29.5 / 17.7, 576 x 576 by 2502 9.3 / 7.2.
// - The chain of a tile where there are few: launch, first loads, stages, epilogue one behind the other while most compute units have nothing.
//   Tiles of 32 x 32 to 64 x 32 whose waves share out the depth give every unit a part, and a residual product of 4096 or more columns is cut along its depth
//   over workgroups (`parts`), whose 32-bit sums meet in memory: the one that arrives last adds them up in the order of the ranges.
// M = 1: dense_gemv.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "common.h"
#include "dense.h"
#include "dense_gemv.h"
#include "device_utils.h"

namespace fh {

constexpr uint32_t ROW_BYTES = 128;
constexpr uint32_t DENSE_RSRC_FLAGS = 0x00020000;   // raw buffer, 32-bit data format
constexpr uint32_t DENSE_K_MAX = 32768;             // a GEMV keeps its vector as floats in LDS

#define FH_LDS3(p) ((__attribute__((address_space(3))) void*)(p))

// LDS of a tile that goes out JP tiles of 32 rows per wave at a time: all of them if they fit in 128 KB.
constexpr uint32_t dense_box(int WN, int WM, int KG, int TN, int JP) { return KG * (32 * TN * WN) * (32 * JP * WM) * 4; }
constexpr int dense_pass(int WN, int WM, int KG, int TN, int TM) { return dense_box(WN, WM, KG, TN, TM) <= 128 * 1024 ? TM : TM / 2; }

template <typename T, int WN, int WM, int KG, int TN, int TM, int NBUF, DenseEpi MODE>
__global__ __launch_bounds__(64 * WN * WM * KG) __attribute__((amdgpu_waves_per_eu(2)))
void dense_gemm_kernel(const T* __restrict__ w, const T* __restrict__ a, uint32_t lda, uint32_t M, uint32_t N, uint32_t K, uint32_t tiles_n,
                       DenseEpiArgs e) {
    extern __shared__ __attribute__((aligned(16))) uint8_t dense_lds[];
    constexpr uint32_t WAVES = WN * WM * KG, BN = 32 * TN * WN, BM = 32 * TM * WM, BK = ROW_BYTES / sizeof(T), ES = sizeof(T), LR = 8 * WAVES;
    constexpr uint32_t BUF = (BN + BM) * ROW_BYTES;
    static_assert(BN % LR == 0 && BM % LR == 0, "every wave has a part of each load");
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t wn = wave % WN, wm = wave / WN % WM, kg = wave / (WN * WM), lrow = lane & 31, lh = lane >> 5;
    // Workgroups go round robin over the 8 XCDs: give each XCD a run of neighbouring tiles (they share operand rows in its L2).
    uint32_t tile = blockIdx.x;
    {
        const uint32_t total = gridDim.x, per = total / 8, x = tile % 8, i = tile / 8;
        if (i < per) tile = x * per + i;          // the last total % 8 tiles stay where they are
    }
    // All tiles of one range of the depth ahead of those of the next: an XCD reads the columns of one or two ranges.
    uint32_t part = 0, st0 = 0, stages = K / BK;
    if (MODE == DenseEpi::Residual && e.parts > 1) {
        const uint32_t tiles = gridDim.x / e.parts, all = stages;
        part = tile / tiles;
        tile -= part * tiles;
        st0 = part * all / e.parts;
        stages = (part + 1) * all / e.parts - st0;
    }
    // Tiles are counted in groups of GROUP rows of tiles, down the column first: the tiles that run at a time share both operands.  512 rows
    // of activations to a group, which an XCD's L2 holds beside the weights (products with a gate, bfloat16, us by 1 / 2 / 4 / 8 rows of tiles:
    // 128 x 128 tiles 3392 x 2048 by 2502 rows 69.0 / 71.8 / 68.0 / 73.9, 6144 x 2048 by 1500 69.7 / 63.5 / 62.7 / 68.2; 128 x 64 tiles
    // 6144 x 2048 by 902 55.8 / 42.3 / 40.9 / 40.9; 256 x 256 tiles 9216 x 3072 by 2502 187.9 / 183.5 / 184.3 / 195.1).
    constexpr uint32_t GROUP = 512 / BM;
    // (One group is one division less ahead of the first loads: 32-bit [gate; up] 3072 x 576 by 65 rows 19.97 us with it, 19.58 without.)
    const uint32_t tiles_m = (M + BM - 1) / BM, first = tiles_m <= GROUP ? 0u : tile / (GROUP * tiles_n) * GROUP, rows = min(GROUP, tiles_m - first), in = tile - first * tiles_n;
    const uint32_t n0 = in / rows * BN, m0 = (first + in % rows) * BM;

    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)(w + (size_t)n0 * K), 0, min(N - n0, BN) * K * ES, DENSE_RSRC_FLAGS);
    const __amdgpu_buffer_rsrc_t ra =
        __builtin_amdgcn_make_buffer_rsrc((void*)(a + (size_t)m0 * lda), 0, ((min(M - m0, BM) - 1) * lda + K) * ES, DENSE_RSRC_FLAGS);
    // load i of wave v fills LDS rows LR i + 8 v .. + 8, lane -> (row, position)
    const uint32_t ld_row = wave * 8 + (lane >> 3);
    const uint32_t ld_piece = (lane & 7) ^ ((ld_row >> 1) & 7);       // rows LR i further on have the same swizzle
    const uint32_t w_off = ld_row * K * ES + ld_piece * 16, a_off = ld_row * lda * ES + ld_piece * 16;
    constexpr uint32_t LOADS = (BN + BM) / LR;
    auto issue = [&](uint32_t stage, uint32_t buf) {
        uint8_t* base = dense_lds + buf * BUF + wave * 1024;
        const uint32_t k = (st0 + stage) * ROW_BYTES;
#pragma unroll
        for (uint32_t i = 0; i < BN / LR; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rw, FH_LDS3(base + i * LR * ROW_BYTES), 16, w_off + i * LR * K * ES, k, 0, 0);
#pragma unroll
        for (uint32_t i = 0; i < BM / LR; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(ra, FH_LDS3(base + (BN + i * LR) * ROW_BYTES), 16, a_off + i * LR * lda * ES, k, 0, 0);
    };
    v16f acc[TN][TM];
#pragma unroll
    for (int i = 0; i < TN; i++)
#pragma unroll
        for (int j = 0; j < TM; j++)
#pragma unroll
            for (int r = 0; r < 16; r++) acc[i][j][r] = 0.f;

    const uint32_t sw = (lrow >> 1) & 7;
    auto frag = [&](const uint8_t* row, uint32_t kk) {
        if constexpr (sizeof(T) == 2) return *reinterpret_cast<const v8bf*>(row + (((2 * kk + lh) ^ sw) * 16));
        else {
            const v4f lo = *reinterpret_cast<const v4f*>(row + (((4 * kk + 2 * lh) ^ sw) * 16));
            const v4f hi = *reinterpret_cast<const v4f*>(row + (((4 * kk + 2 * lh + 1) ^ sw) * 16));
            return (v8f){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        }
    };
    // The next stage's tiles are in LDS (those of the stages after it may still be on their way), and every wave is done with this one's.
    // Two buffers: the compiler's own wait, around which it moves the next fragments' reads (32-bit 2048 x 8192 by 130 rows 161.8 us behind a wait
    // in assembly, 159.0 this way; 576 x 576 by 64 with two norms 18.2 / 17.4).
    auto arrive = [&](bool last) {
        if constexpr (NBUF == 2) {
            __builtin_amdgcn_s_waitcnt(0);
            __syncthreads();
        } else {
            if (!last) asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"((NBUF - 2) * LOADS) : "memory");
            else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
    };
#pragma unroll
    for (uint32_t st = 0; st < NBUF - 1; st++)
        if (st < stages) issue(st, st);
    arrive(stages < NBUF - 1);
    uint32_t buf = 0;
    for (uint32_t st = 0; st < stages; st++) {
        const uint32_t ahead = st + NBUF - 1;
        if (ahead < stages) issue(ahead, buf == 0 ? NBUF - 1 : buf - 1);
        const uint8_t* wb = dense_lds + buf * BUF + (wn * 32 * TN + lrow) * ROW_BYTES;
        const uint8_t* ab = dense_lds + buf * BUF + (BN + wm * 32 * TM + lrow) * ROW_BYTES;
#pragma unroll
        for (uint32_t k = 0; k < BK / 16 / KG; k++) {
            const uint32_t kk = kg * (BK / 16 / KG) + k;
            typename Vec<T>::x8 fw[TN], fa[TM];
#pragma unroll
            for (int i = 0; i < TN; i++) fw[i] = frag(wb + i * 32 * ROW_BYTES, kk);
#pragma unroll
            for (int j = 0; j < TM; j++) fa[j] = frag(ab + j * 32 * ROW_BYTES, kk);
#pragma unroll
            for (int i = 0; i < TN; i++)
#pragma unroll
                for (int j = 0; j < TM; j++) acc[i][j] = mma32(fw[i], fa[j], acc[i][j]);
        }
        arrive(ahead >= stages);
        buf = buf == NBUF - 1 ? 0 : buf + 1;
    }
    // The tile goes through LDS, so that a row's neighbouring columns are written (and read) by neighbouring lanes; the waves that shared
    // out the depth of a tile meet there.  The 16-byte piece c of row r sits at c ^ (r & 7): no bank conflicts either way.
    constexpr int JP = dense_pass(WN, WM, KG, TN, TM);
    constexpr uint32_t THREADS = 64 * WAVES, ROWS = 32 * JP * WM, PIECES = BN / 4, STEP = THREADS / PIECES, STEPS = ROWS / STEP, G = STEPS < 4 ? STEPS : 4;
    static_assert(THREADS % PIECES == 0 && ROWS % STEP == 0 && STEPS % G == 0, "whole steps");
    v4f* box = reinterpret_cast<v4f*>(dense_lds);
    const uint32_t piece = tid % PIECES, n = n0 + 4 * piece;
    const EpiCols<MODE> cols = n < N ? epilogue_cols<MODE>(e, n) : EpiCols<MODE>{};
#pragma unroll
    for (uint32_t p = 0; p < TM / JP; p++) {
        if (p > 0) __syncthreads();
#pragma unroll
        for (int i = 0; i < TN; i++)
#pragma unroll
            for (int j = 0; j < JP; j++)
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const v16f& c = acc[i][p * JP + j];
                    const uint32_t r = (wm * JP + j) * 32 + lrow, at = (wn * TN + i) * 8 + 2 * g + lh;
                    box[(kg * ROWS + r) * PIECES + (at ^ (r & 7))] = (v4f){c[4 * g], c[4 * g + 1], c[4 * g + 2], c[4 * g + 3]};
                }
        __syncthreads();
        if constexpr (MODE == DenseEpi::Residual && JP == TM)
            if (e.parts > 1) {
                // Stores and loads past the caches of an XCD, 8 bytes a lane in two planes.  A wave's stores have arrived before the barrier that lets the
                // workgroup count itself in; who counts `parts` sees them all, and leaves the counter at zero for the next launch.
                constexpr uint32_t PLANE = ROWS * PIECES;
                uint64_t* mine = e.sums + (size_t)(tile * e.parts + part) * (2 * PLANE);
#pragma unroll
                for (uint32_t s = 0; s < STEPS; s++) {
                    const uint32_t r = s * STEP + tid / PIECES, at = r * PIECES + piece;
                    if (n >= N || m0 + r >= M) continue;
                    v4f v = box[r * PIECES + (piece ^ (r & 7))];
#pragma unroll
                    for (int k = 1; k < KG; k++) v += box[(k * ROWS + r) * PIECES + (piece ^ (r & 7))];
                    uint64_t h[2];
                    __builtin_memcpy(h, &v, 16);
                    __hip_atomic_store(mine + at, h[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    __hip_atomic_store(mine + PLANE + at, h[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                __shared__ uint32_t arrived;
                __syncthreads();
                if (tid == 0) {
                    arrived = __hip_atomic_fetch_add(e.arrivals + tile, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
                    if (arrived == e.parts) __hip_atomic_store(e.arrivals + tile, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                }
                __syncthreads();
                if (arrived != e.parts || n >= N) return;
                const uint64_t* from = e.sums + (size_t)tile * e.parts * (2 * PLANE);
#pragma unroll
                for (uint32_t s0 = 0; s0 < STEPS; s0 += G) {
                    EpiRow<T, MODE> row[G];
                    v4f v[G];
#pragma unroll
                    for (uint32_t s = 0; s < G; s++) {
                        const uint32_t m = m0 + (s0 + s) * STEP + tid / PIECES;
                        v[s] = (v4f){0.f, 0.f, 0.f, 0.f};
                        if (m < M) row[s] = epilogue_row<T, MODE>(e, m, n);
                    }
                    for (uint32_t q = 0; q < e.parts; q++) {
                        uint64_t h[G][2];
#pragma unroll
                        for (uint32_t s = 0; s < G; s++) {
                            const uint32_t r = min((s0 + s) * STEP + tid / PIECES, M - 1 - m0);      // rows past the end: what another lane adds up
                            const uint64_t* at = from + (size_t)q * (2 * PLANE) + r * PIECES + piece;
                            h[s][0] = __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                            h[s][1] = __hip_atomic_load(at + PLANE, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                        }
#pragma unroll
                        for (uint32_t s = 0; s < G; s++) {
                            v4f x;
                            __builtin_memcpy(&x, h[s], 16);
                            v[s] += x;
                        }
                    }
#pragma unroll
                    for (uint32_t s = 0; s < G; s++) {
                        const uint32_t m = m0 + (s0 + s) * STEP + tid / PIECES;
                        const float f[4] = {v[s][0], v[s][1], v[s][2], v[s][3]};
                        if (m < M) dense_epilogue<T, MODE>(e, m, n, N, f, cols, row[s]);
                    }
                }
                return;
            }
        if (n >= N) continue;
#pragma unroll
        for (uint32_t s0 = 0; s0 < STEPS; s0 += G) {
            EpiRow<T, MODE> row[G];
            uint32_t m[G];
            v4f v[G];
#pragma unroll
            for (uint32_t s = 0; s < G; s++) {
                const uint32_t r = (s0 + s) * STEP + tid / PIECES;
                m[s] = m0 + ((r / (32 * JP)) * TM + p * JP) * 32 + r % (32 * JP);
                if (m[s] < M) row[s] = epilogue_row<T, MODE>(e, m[s], n);
                v[s] = box[r * PIECES + (piece ^ (r & 7))];
#pragma unroll
                for (int k = 1; k < KG; k++) v[s] += box[(k * ROWS + r) * PIECES + (piece ^ (r & 7))];
            }
#pragma unroll
            for (uint32_t s = 0; s < G; s++)
                if (m[s] < M) {
                    const float f[4] = {v[s][0], v[s][1], v[s][2], v[s][3]};
                    dense_epilogue<T, MODE>(e, m[s], n, N, f, cols, row[s]);
                }
        }
    }
}

// The vector of a one-row product goes into LDS as floats, made from what DenseIn names.
template <typename T, int KS, DenseEpi MODE, DenseIn::Kind IN, int STEPS>
__global__ __launch_bounds__(GEMV_THREADS) void dense_gemv_kernel(const T* __restrict__ w, DenseIn in, uint32_t N, uint32_t K, DenseEpiArgs e) {
    extern __shared__ __attribute__((aligned(16))) float gemv_lds[];
    const uint32_t tid = threadIdx.x;
    float* xs = gemv_lds;
    float* red = gemv_lds + K;
    typedef typename Vec<T>::x4 x4;
    typedef typename Vec<T>::x8 x8;
    // What the prologue reads first is requested ahead of the matrix, into registers: NV pieces per thread of 4 columns (Rows: 8).
    constexpr uint32_t NV = STEPS == 1 ? 1 : 3;
    if constexpr (IN == DenseIn::Rows) {
        const T* a = (const T*)in.rows;
        x8 v[NV];
#pragma unroll
        for (uint32_t i = 0; i < NV; i++) {
            const uint32_t k = (tid + i * GEMV_THREADS) * 8;
            if (k < K) v[i] = load8(a + k);
        }
        gemv_body<T, KS, MODE, STEPS>(w, N, K, blockIdx.x * gemv_rows<KS>(), xs, red, e, [&]() {
            auto put = [&](uint32_t k, const x8& x) {
#pragma unroll
                for (int j = 0; j < 8; j++) xs[k + j] = (float)x[j];
            };
#pragma unroll
            for (uint32_t i = 0; i < NV; i++) {
                const uint32_t k = (tid + i * GEMV_THREADS) * 8;
                if (k < K) put(k, v[i]);
            }
            for (uint32_t k = (tid + NV * GEMV_THREADS) * 8; k < K; k += GEMV_THREADS * 8) put(k, load8(a + k));
        });
    } else if constexpr (IN == DenseIn::Normed) {
        v4f v[NV], lw[NV], lb[NV];
#pragma unroll
        for (uint32_t i = 0; i < NV; i++) {
            const uint32_t k = (tid + i * GEMV_THREADS) * 4;
            v[i] = (v4f){0.f, 0.f, 0.f, 0.f};
            if (k < K) {
                v[i] = *reinterpret_cast<const v4f*>(in.f32 + k);
                lw[i] = *reinterpret_cast<const v4f*>(in.ln.w + k);
                lb[i] = *reinterpret_cast<const v4f*>(in.ln.b + k);
            }
        }
        gemv_body<T, KS, MODE, STEPS>(w, N, K, blockIdx.x * gemv_rows<KS>(), xs, red, e, [&]() {
            // a thread keeps to its own elements until the product's barrier; those past the registers wait in LDS
            constexpr uint32_t REST = NV * GEMV_THREADS * 4;
            float s = 0.f;
#pragma unroll
            for (uint32_t i = 0; i < NV; i++) s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);      // zero past ln.n
            for (uint32_t k = REST + tid * 4; k < K; k += GEMV_THREADS * 4) {
                const v4f x = *reinterpret_cast<const v4f*>(in.f32 + k);
                *reinterpret_cast<v4f*>(xs + k) = x;
                s += (x[0] + x[1]) + (x[2] + x[3]);
            }
            const float mean = block_sum(s, red, tid, GEMV_THREADS) / (float)in.ln.n;
            float ss = 0.f;
            auto square = [&](uint32_t k, const v4f& x) {
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const float d = x[j] - mean;
                    if (k + j < in.ln.n) ss = fmaf(d, d, ss);
                }
            };
#pragma unroll
            for (uint32_t i = 0; i < NV; i++) square((tid + i * GEMV_THREADS) * 4, v[i]);
            for (uint32_t k = REST + tid * 4; k < K; k += GEMV_THREADS * 4) square(k, *reinterpret_cast<const v4f*>(xs + k));
            const float inv = 1.0f / sqrtf(block_sum(ss, red, tid, GEMV_THREADS) / (float)in.ln.n + in.ln.eps);
            auto put = [&](uint32_t k, const v4f& x, const v4f& nw, const v4f& nb) {
                v4f y;
#pragma unroll
                for (int j = 0; j < 4; j++) y[j] = (x[j] - mean) * inv * nw[j] + nb[j];
                *reinterpret_cast<v4f*>(xs + k) = y;
            };
#pragma unroll
            for (uint32_t i = 0; i < NV; i++) {
                const uint32_t k = (tid + i * GEMV_THREADS) * 4;
                if (k < K) put(k, v[i], lw[i], lb[i]);
            }
            for (uint32_t k = REST + tid * 4; k < K; k += GEMV_THREADS * 4)
                put(k, *reinterpret_cast<const v4f*>(xs + k), *reinterpret_cast<const v4f*>(in.ln.w + k), *reinterpret_cast<const v4f*>(in.ln.b + k));
        });
    } else {
        // head = a multiple of 32 columns: lane group of 16, 4 columns per lane and step; the first head's first 128 columns in registers
        constexpr uint32_t NH = 2;
        const uint32_t h0 = tid / 16, c0 = tid % 16 * 4;
        v4f v0[NH], hw0[NH];
        x4 g0[NH];
#pragma unroll
        for (uint32_t i = 0; i < NH; i++) {
            const uint32_t c = c0 + 64 * i;
            v0[i] = (v4f){0.f, 0.f, 0.f, 0.f};
            if (h0 < in.heads && c < in.head) {
                v0[i] = *reinterpret_cast<const v4f*>(in.f32 + h0 * in.head + c);
                hw0[i] = *reinterpret_cast<const v4f*>(in.w + c);
                g0[i] = *reinterpret_cast<const x4*>((const T*)in.gate + h0 * in.head + c);
            }
        }
        gemv_body<T, KS, MODE, STEPS>(w, N, K, blockIdx.x * gemv_rows<KS>(), xs, red, e, [&]() {
            const uint32_t n = in.heads * in.head;
            for (uint32_t k = n + tid; k < K; k += GEMV_THREADS) xs[k] = 0.f;
            for (uint32_t h = h0; h < in.heads; h += GEMV_THREADS / 16) {
                const float* o = in.f32 + h * in.head;
                float ss = 0.f;
                auto square = [&](const v4f& v) {
#pragma unroll
                    for (int j = 0; j < 4; j++) ss = fmaf(v[j], v[j], ss);      // zero past head_n
                };
                const bool first = h == h0;
                if (first) {
#pragma unroll
                    for (uint32_t i = 0; i < NH; i++) square(v0[i]);
                }
                for (uint32_t c = c0 + (first ? 64 * NH : 0); c < in.head; c += 64) square(*reinterpret_cast<const v4f*>(o + c));
                ss = lane_xor_add<8>(ss); ss = lane_xor_add<4>(ss); ss = lane_xor_add<2>(ss); ss = lane_xor_add<1>(ss);
                const float inv = 1.0f / sqrtf(ss / (float)in.head_n + in.eps);
                auto put = [&](uint32_t c, const v4f& v, const v4f& hw, const x4& g) {
#pragma unroll
                    for (int j = 0; j < 4; j++) xs[h * in.head + c + j] = v[j] * inv * hw[j] * (float)g[j];
                };
                if (first) {
#pragma unroll
                    for (uint32_t i = 0; i < NH; i++)
                        if (c0 + 64 * i < in.head) put(c0 + 64 * i, v0[i], hw0[i], g0[i]);
                }
                for (uint32_t c = c0 + (first ? 64 * NH : 0); c < in.head; c += 64)
                    put(c, *reinterpret_cast<const v4f*>(o + c), *reinterpret_cast<const v4f*>(in.w + c), *reinterpret_cast<const x4*>((const T*)in.gate + h * in.head + c));
            }
        });
    }
}

// One workgroup per row; a thread holds NV groups of four elements.
template <typename T, int NV>
__global__ __launch_bounds__(256) void layer_norm_kernel(const float* __restrict__ x, uint32_t ldx, LayerNorm ln, uint32_t width, T* __restrict__ out, uint32_t ld_out) {
    __shared__ float red[4];
    const uint32_t m = blockIdx.x, tid = threadIdx.x;
    v4f v[NV];
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const uint32_t c = (tid + 256 * i) * 4;
        v[i] = c < width ? *reinterpret_cast<const v4f*>(x + (size_t)m * ldx + c) : (v4f){0.f, 0.f, 0.f, 0.f};
        s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);                  // zero past ln.n
    }
    const float mean = block_sum(s, red, tid, 256) / (float)ln.n;
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < NV; i++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float d = v[i][j] - mean;
            if ((tid + 256 * i) * 4 + j < ln.n) ss = fmaf(d, d, ss);
        }
    const float inv = 1.0f / sqrtf(block_sum(ss, red, tid, 256) / (float)ln.n + ln.eps);
#pragma unroll
    for (int i = 0; i < NV; i++) {
        const uint32_t c = (tid + 256 * i) * 4;
        if (c >= width) continue;
        const v4f w = *reinterpret_cast<const v4f*>(ln.w + c), b = *reinterpret_cast<const v4f*>(ln.b + c);
        float y[4];
#pragma unroll
        for (int j = 0; j < 4; j++) y[j] = (v[i][j] - mean) * inv * w[j] + b[j];
        store4<T>(out + (size_t)m * ld_out + c, y[0], y[1], y[2], y[3]);
    }
}

template <typename T>
__global__ __launch_bounds__(256) void dense_embedding_kernel(const T* __restrict__ table, uint32_t ld_table, uint32_t width, float scale, const uint32_t* __restrict__ tokens,
                                                              float* __restrict__ x, uint32_t ldx, DynTanh next, T* __restrict__ out, uint32_t ld_out,
                                                              T* __restrict__ out2, uint32_t ld_out2, uint32_t* __restrict__ counts) {
    const uint32_t m = blockIdx.y, tok = tokens[m], i = blockIdx.x * 256 + threadIdx.x;
    if (i < ldx) {
        const float v = i < width ? (float)table[(size_t)tok * ld_table + i] * scale : 0.f;
        x[(size_t)m * ldx + i] = v;
        if (out) out[(size_t)m * ld_out + i] = (T)dyn_tanh(next, i, v);
        if (out2) out2[(size_t)m * ld_out2 + i] = (T)v;
    }
    if (i == 0 && counts) atomicAdd(counts + tok, 1u);
}

template <typename T>
__global__ __launch_bounds__(256) void gather_rows_kernel(const T* __restrict__ a, uint32_t lda, const uint32_t* __restrict__ rows, uint32_t width,
                                                          T* __restrict__ out, uint32_t ld_out) {
    const T* src = a + (size_t)rows[blockIdx.x] * lda;
    for (uint32_t i = threadIdx.x; i < width; i += blockDim.x) out[(size_t)blockIdx.x * ld_out + i] = src[i];
}

namespace {

template <typename T, int WN, int WM, int KG, int TN, int TM, int NBUF, DenseEpi MODE, bool RANGES = false>
void go_gemm(const DenseWeight& w, const void* a, uint32_t lda, uint32_t M, const DenseEpiArgs& e, hipStream_t s, uint32_t ranges = 1) {
    static_assert(!RANGES || (MODE == DenseEpi::Residual && dense_pass(WN, WM, KG, TN, TM) == TM), "ranges of the depth meet in an epilogue of one pass");
    const uint32_t parts = RANGES ? ranges : 1;
    constexpr uint32_t BN = 32 * TN * WN, BM = 32 * TM * WM, stage = (BN + BM) * ROW_BYTES * NBUF, box = dense_box(WN, WM, KG, TN, dense_pass(WN, WM, KG, TN, TM)),
                       lds = stage > box ? stage : box;
    const auto kernel = dense_gemm_kernel<T, WN, WM, KG, TN, TM, NBUF, MODE>;
    static const hipError_t lds_ok = hipFuncSetAttribute((const void*)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    (void)lds_ok;
    const uint32_t tn = (w.N + BN - 1) / BN, tm = (M + BM - 1) / BM;
    DenseEpiArgs args = e;
    args.parts = parts;
    fh::launch(kernel, dim3(tn * tm * parts), 64 * WN * WM * KG, lds, s, (const T*)w.p, (const T*)a, lda, M, w.N, w.K, tn, args);
}

template <typename T, int KS, DenseEpi MODE, DenseIn::Kind IN, int STEPS>
void gemv_steps(const DenseWeight& w, const DenseIn& in, const DenseEpiArgs& e, hipStream_t s) {
    static const hipError_t lds_ok = hipFuncSetAttribute((const void*)dense_gemv_kernel<T, KS, MODE, IN, STEPS>, hipFuncAttributeMaxDynamicSharedMemorySize, (DENSE_K_MAX + 16) * 4);
    (void)lds_ok;
    fh::launch(dense_gemv_kernel<T, KS, MODE, IN, STEPS>, dim3((w.N + gemv_rows<KS>() - 1) / gemv_rows<KS>()), GEMV_THREADS, (w.K + 16) * 4, s, (const T*)w.p,
               in, w.N, w.K, e);
}

template <typename T, int KS, DenseEpi MODE, DenseIn::Kind IN>
void go_gemv(const DenseWeight& w, const DenseIn& in, const DenseEpiArgs& e, hipStream_t s) {
    if (w.K <= gemv_step<T, KS>()) gemv_steps<T, KS, MODE, IN, 1>(w, in, e, s);
    else gemv_steps<T, KS, MODE, IN, 2>(w, in, e, s);
}

template <typename T, DenseEpi MODE, DenseIn::Kind IN>
void go_row(const DenseWeight& w, const DenseIn& in, const DenseEpiArgs& e, hipStream_t s) {
    switch (gemv_depth_split(w.N, w.K)) {
        case 1: go_gemv<T, 1, MODE, IN>(w, in, e, s); return;
        case 2: go_gemv<T, 2, MODE, IN>(w, in, e, s); return;
        default: go_gemv<T, 4, MODE, IN>(w, in, e, s); return;
    }
}

template <typename T, DenseEpi MODE>
void go(const DenseWeight& w, const DenseIn& in, uint32_t M, const DenseEpiArgs& e, hipStream_t s) {
    if (M == 1) {
        if constexpr (MODE == DenseEpi::RawGate || MODE == DenseEpi::ActPair)
            if (in.kind == DenseIn::Normed) { go_row<T, MODE, DenseIn::Normed>(w, in, e, s); return; }
        if constexpr (MODE == DenseEpi::Residual)
            if (in.kind == DenseIn::HeadGate) { go_row<T, MODE, DenseIn::HeadGate>(w, in, e, s); return; }
        if constexpr (MODE != DenseEpi::Rope && MODE != DenseEpi::Split && MODE != DenseEpi::GateMul) { go_row<T, MODE, DenseIn::Rows>(w, in, e, s); return; }
    }
    const void* a = in.rows;
    const uint32_t lda = in.lda;
    auto tiles = [&](uint32_t bn, uint32_t bm) { return (uint64_t)((w.N + bn - 1) / bn) * ((M + bm - 1) / bm); };
    constexpr uint64_t CUS = 256;
    if constexpr (sizeof(T) == 2) {
        // Up to a few tiles of 32 rows a compute unit: the smallest tiles, four waves to the depth of each (us, by the rules below / 32 x 32 / 64 x 32, columns
        // first; o, down: residual products with two norms): gate 928 x 576 by 65 rows 6.5 / 3.8 / 4.8, by 300 6.5 / 4.2 / 5.0, by 902 (841 and 435 tiles)
        // 8.3 / 6.1 / 6.2, o 576 x 576 by 300 9.1 / 5.0 / 6.7, by 902 (522) 10.9 / 6.9 / 8.1, down 576 x 1536 by 902 13.3 / 10.9 / 12.7, up 3072 x 576 by 300
        // (960 and 480) 7.8 / 6.3 / 5.8, gate 6272 x 2048 by 130 (980 and 490) 17.7 / 14.6 / 11.7.  Past that the operands' traffic counts: up 16384 x 2048 by 33
        // (1024 and 512) 17.9 / 20.2 / 19.4, 2048 x 2048 by 902 rows (1856 and 928) 16.3 / 25.3 / 21.3.  Shallow residual products end in two hyperbolic tangents an
        // element and gain by more workgroups a little longer (32 columns x 64 rows, 720 tiles: o by 2502 rows 13.0 / 10.5, down 17.8 / 17.1).
        const uint64_t t64 = tiles(64, 64), t6432 = tiles(64, 32), t128 = tiles(128, 128);
        if constexpr (MODE == DenseEpi::Residual) {
            // Deep ones in ranges of the depth, us for 2048 x 8192 before / by 64 x 32 x 8 ranges / 64 x 64 x 4 / 128 x 128 x as many as give every compute unit one:
            // by 5 rows 35 / 11.7 / 14.6 / 20.8, by 33 35 / 13.5 / 15.9 / 21.4, by 65 35 / 16.4 / 16.2 / 22.2, by 200 36 / - / 22.1 / 24.4, by 300 37 / - / 33.3 / 25.9,
            // by 500 38 / - / - / 31.5, by 902 59 / - / - / 44.9.
            if (w.K >= 4096 && e.sums) {
                const uint32_t large = t128 <= CUS / 2 ? (uint32_t)std::min<uint64_t>(8, CUS / t128) : 1;
                if (t6432 <= 80) { go_gemm<T, 1, 1, 4, 2, 1, 4, MODE, true>(w, a, lda, M, e, s, 8); return; }
                if (t64 <= CUS / 2) { go_gemm<T, 1, 1, 4, 2, 2, 4, MODE, true>(w, a, lda, M, e, s, 4); return; }
                if (large > 1) { go_gemm<T, 2, 2, 2, 2, 2, 3, MODE, true>(w, a, lda, M, e, s, large); return; }
            }
        }
        if (tiles(32, 32) <= 3 * CUS) { go_gemm<T, 1, 1, 4, 1, 1, 4, MODE>(w, a, lda, M, e, s); return; }
        if (t6432 < 2 * CUS) { go_gemm<T, 1, 1, 4, 2, 1, 4, MODE>(w, a, lda, M, e, s); return; }
        if constexpr (MODE == DenseEpi::Residual)
            if (w.K < 2048 && tiles(32, 64) <= 3 * CUS) { go_gemm<T, 1, 2, 2, 1, 1, 4, MODE>(w, a, lda, M, e, s); return; }
        // The largest tile that keeps the chip busy (us, 256 x 256 / 128 x 128 / 128 x 64 / 64 x 64; gate: input products, up: gate and up,
        // res: residual products of a prompt):
        // - 256 x 256, one workgroup a compute unit, if its last round is at least 0.8 full on average: up 16384 x 2048 by 902 rows (256 tiles)
        //   66.0 / 70.6 / 83 / 92, gate 6144 x 2048 by 2502 (240) 70.1 / 70.5 / 85 / 92, by 902 (96) 59.2 / 35.1 / 37.3 / 42.9.  Not for up to 128
        //   rows, of which it would compute 256: 128256 x 2048 by 128 148 / 138 / 148 / 164, by 200 162 / 182 / 211 / 243.
        // - 128 x 128, two workgroups a compute unit, from more than one on: res 2048 x 2048 by 2502 (320) 54 / 31.4 / 36.9 / 39.8, up
        //   3072 x 576 by 2502 (480) 25.7 / 16.3 / 19.2 / 18.8; one on each, 16384 x 2048 by 130 (256): 46 / 25.0 / 21.0 / 20.2.  Eight waves to a
        //   tile: four, with two 32 x 32 tiles more each, do not cover the gate's exponentials and the stores (gate 3392 x 2048 by 2502 rows 62.0
        //   with four, 57.1 with eight, res 2048 x 8192 by 2502 106.2 / 99.3, gate 9216 x 3072 by 2502 151.7 / 148.0).
        // - 64 x 64 where two a compute unit hold all of them: res 2048 x 8192 by 902 (480) 159 / 76 / 49.7 / 46.6, gate 6144 x 2048 by 300 (480)
        //   56 / 26 / 16.8 / 16.0; and for up to 64 rows, of which the others would compute 128: 128256 x 2048 by 2 118 / 103 / 96 / 91, by 64
        //   135 / 122 / 117 / 119, 49152 x 576 by 2 16.6 / 11.0 / 11.0 / 9.9.
        //   Deep ones are a chain of stages: four buffers and a quarter of the depth for each wave against two buffers and a quarter of the tile:
        //   res 2048 x 8192 by 130 rows 35.0 / 59.2, 2048 x 2048 by 520 14.3 / 18.1, but gate 1152 x 576 by 902 8.2 / 7.5.  The shallow form
        //   wins up to four on a compute unit: gate 928 x 576 by 2502 rows (600) 33 / 12.9 / 10.7 / 9.2, up 3072 x 576 by 1344 (1008) - / 12.7 / 11.2 /
        //   11.2, but gate 1728 x 576 by 2502 (1080) 33 / 14.9 / 17.0 / 15.6, up 3072 x 576 by 1500 (1152) 25 / 13.0 / 15.4 / 15.3.
        const uint64_t t256 = tiles(256, 256), rounds = (t256 + CUS - 1) / CUS;
        const bool deep = w.K >= 1024, small = M <= 64 || t64 <= 2 * CUS || (!deep && t64 <= 4 * CUS);
        if (small && deep) go_gemm<T, 1, 1, 4, 2, 2, 4, MODE>(w, a, lda, M, e, s);
        else if (small) go_gemm<T, 2, 2, 1, 1, 1, 2, MODE>(w, a, lda, M, e, s);
        else if (M > 128 && 5 * t256 >= 4 * CUS * rounds) go_gemm<T, 4, 2, 1, 2, 4, 2, MODE>(w, a, lda, M, e, s);
        else if (t128 > CUS) go_gemm<T, 4, 2, 1, 1, 2, 2, MODE>(w, a, lda, M, e, s);
        else go_gemm<T, 2, 2, 2, 2, 1, 3, MODE>(w, a, lda, M, e, s);
    } else {
        // 32-bit: bound by the matrix unit's rate; the large tile when its tiles give most compute units work, small ones (as above, two waves to the depth) when
        // 64 x 64 leave most of them idle: us by 64 x 64 / 32 x 32 / 32 x 64 / 64 x 32, columns first: o 576 x 576 by 300 rows (180 tiles of 32 x 32) 16.8 / 10.3 / 11.0 / 11.7, by 700 (396) 17.5 /
        // 14.8 / 11.7 / 12.3, up 3072 x 576 by 130 (288 and 240) 15.6 / 12.7 / 13.2 / 10.5, down 576 x 1536 by 20 32.9 / 20.6 / 21.5 / 22.5, up by 700 (1056 and 1056) 31.8 with
        // 128 x 128 tiles / 34.8 / 28.7 / 29.6.
        if (tiles(32, 32) <= CUS) go_gemm<T, 1, 1, 2, 1, 1, 4, MODE>(w, a, lda, M, e, s);
        else if (tiles(64, 32) <= CUS) go_gemm<T, 2, 1, 2, 1, 1, 4, MODE>(w, a, lda, M, e, s);
        else if (tiles(32, 64) <= 5 * CUS) go_gemm<T, 1, 2, 2, 1, 1, 4, MODE>(w, a, lda, M, e, s);
        else if (tiles(128, 128) >= 192) go_gemm<T, 2, 2, 1, 2, 2, 2, MODE>(w, a, lda, M, e, s);
        else go_gemm<T, 2, 2, 1, 1, 1, 2, MODE>(w, a, lda, M, e, s);
    }
}

template <typename T>
void by_mode(const DenseWeight& w, const DenseIn& in, uint32_t M, DenseEpi mode, const DenseEpiArgs& e, hipStream_t s) {
    switch (mode) {
        case DenseEpi::F32: go<T, DenseEpi::F32>(w, in, M, e, s); break;
        case DenseEpi::RawGate: go<T, DenseEpi::RawGate>(w, in, M, e, s); break;
        case DenseEpi::Rope: go<T, DenseEpi::Rope>(w, in, M, e, s); break;
        case DenseEpi::Split: go<T, DenseEpi::Split>(w, in, M, e, s); break;
        case DenseEpi::GateMul: go<T, DenseEpi::GateMul>(w, in, M, e, s); break;
        case DenseEpi::ActPair: go<T, DenseEpi::ActPair>(w, in, M, e, s); break;
        case DenseEpi::Residual: go<T, DenseEpi::Residual>(w, in, M, e, s); break;
    }
}

}  // namespace

uint32_t dense_k_max() { return DENSE_K_MAX; }
// At most 640 tiles and ranges of 64 x 32 results, 512 of 64 x 64 or 256 of 128 x 128; at most 128 tiles.
size_t dense_sums_bytes() { return (size_t)256 * 128 * 128 * 4; }
size_t dense_arrivals_bytes() { return 128 * 4; }

void launch_dense(DType t, const DenseWeight& w, const DenseIn& in, uint32_t M, DenseEpi mode, const DenseEpiArgs& e, hipStream_t s) {
    if (M == 0 || w.N == 0) return;
    if (t == DType::BF16) by_mode<__bf16>(w, in, M, mode, e, s);
    else by_mode<float>(w, in, M, mode, e, s);
}

namespace {

template <typename T>
void layer_norm(const float* x, uint32_t ldx, const LayerNorm& ln, uint32_t width, uint32_t M, void* out, uint32_t ld_out, hipStream_t s) {
    auto go = [&](auto kernel) { fh::launch(kernel, dim3(M), 256, 0, s, x, ldx, ln, width, (T*)out, ld_out); };
    if (width <= 1024) go(layer_norm_kernel<T, 1>);
    else if (width <= 2048) go(layer_norm_kernel<T, 2>);
    else if (width <= 4096) go(layer_norm_kernel<T, 4>);
    else go(layer_norm_kernel<T, 16>);
}

}  // namespace

void launch_layer_norm(DType t, const float* x, uint32_t ldx, const LayerNorm& ln, uint32_t width, uint32_t M, void* out, uint32_t ld_out, hipStream_t s) {
    if (t == DType::BF16) layer_norm<__bf16>(x, ldx, ln, width, M, out, ld_out, s);
    else layer_norm<float>(x, ldx, ln, width, M, out, ld_out, s);
}

void launch_dense_embedding(DType t, const void* table, uint32_t ld_table, uint32_t width, float scale, const uint32_t* tokens_dev, uint32_t M, float* x,
                            uint32_t ldx, const DynTanh& next, void* out, uint32_t ld_out, void* out2, uint32_t ld_out2, uint32_t* counts, hipStream_t s) {
    if (t == DType::BF16)
        fh::launch(dense_embedding_kernel<__bf16>, dim3((ldx + 255) / 256, M), 256, 0, s, (const __bf16*)table, ld_table, width, scale, tokens_dev, x, ldx, next, (__bf16*)out, ld_out,
                   (__bf16*)out2, ld_out2, counts);
    else
        fh::launch(dense_embedding_kernel<float>, dim3((ldx + 255) / 256, M), 256, 0, s, (const float*)table, ld_table, width, scale, tokens_dev, x, ldx, next, (float*)out, ld_out,
                   (float*)out2, ld_out2, counts);
}

void launch_gather_rows(DType t, const void* a, uint32_t lda, const uint32_t* rows_dev, uint32_t n, uint32_t width, void* out, uint32_t ld_out, hipStream_t s) {
    if (t == DType::BF16) fh::launch(gather_rows_kernel<__bf16>, dim3(n), 256, 0, s, (const __bf16*)a, lda, rows_dev, width, (__bf16*)out, ld_out);
    else fh::launch(gather_rows_kernel<float>, dim3(n), 256, 0, s, (const float*)a, lda, rows_dev, width, (float*)out, ld_out);
}

}  // namespace fh
