// Quantised matmul for a few rows of activations (matmul_mat_q8_0_KxN / matmul_mat_q4_0_KxN, emit.rs:2108-2302, 3667-3817), fast
// mode: what a short prompt, or a handful of sequences side by side, multiplies.
//
// What bounds it: the weights' way from memory (each byte is used for a few rows only) and latency.  The tile kernel (gemm.hip) walks
// the whole of K in one workgroup of 128 columns, about 1.1 us per 128-deep stage however few rows there are, on N / 128 workgroups.
// Here a workgroup takes a 32 x 32 tile, or two of the same columns (twice that with the SiLU epilogue), and its waves share out K, each through a strip of LDS of its own:
// no barrier until the waves' partial tiles meet at the end, where they are added in the order of K.
// Block sums are exact (v_mfma_i32_32x32x32_i8, one quant block per instruction); the scales' products come from a rank-1
// v_mfma_f32_32x32x8_f16, exact in f32.  Up to a depth of 4096 a block's sum is converted and added with one FMA: an error of 2e-7 of the
// typical output, and with so few rows no slower than the tile kernel's biased sums (2e-5).  Deeper sums are biased (BIASED): there
// that kernel's own rounding reaches 1e-4 of a result, and a row would differ by all of it between a small and a large batch.
// 32 rows of 2048 -> 8192: 6.2 us (2.7 TB/s of weights) against the tile kernel's 22; 8192 -> 2048: 12.5 against 76 (22 with K ranges);
// [gate; up] with its epilogue, 2048 -> 16384: 10.5 against 29.5.  Operands fetched straight into registers took 10 and 31 us.
// The scales' arithmetic is half of a wave's work (16 conversions and FMAs a block and tile), so rows of padding are left out by groups of 8: 2048 -> 8192 by 37 rows 10.7 -> 10.3 us with the
// quantiser, Q8_0 11.5 -> 10.9, 3072 -> 8192 13.5 -> 12.8, 8192 -> 2048 by 8 Q8_0 15.0 -> 14.0.
#include <stdlib.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "common.h"
#include "device_utils.h"

namespace fh {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef _Float16 v8h __attribute__((ext_vector_type(8)));

constexpr int FR_U = 4;                      // blocks of a step: 128 bytes of a Q8_0 or activation row, 64 of a Q4_0 row
constexpr int FR_AGENT = 16;                 // a load past this XCD's L2 (SC1)
constexpr uint32_t FR_RSRC = 0x00020000;     // raw buffer, 32-bit data format
constexpr uint32_t FR_MAGIC = 0x4B400000u;   // 12582912.0f: the bias that makes a block sum a float (gemm.hip)
constexpr int FR_A_LOG2 = 8;                 // its removal: activation scales times 2^8, weight scales times 2^15 and 2^14

struct FewArgs {
    const uint8_t* wq;
    const uint16_t* wsc;
    const int8_t* aq;            // odd blocks negated, as for the tile kernel
    const uint16_t* asc;
    float* y;
    uint32_t M, N, K, ldy, accumulate;
    int8_t* silu_q;              // SILU: [M][inter] codes (odd blocks negated), [M][inter / 32] scales
    uint16_t* silu_sc;
    uint32_t inter;
    // RAW: the activations as they come; a workgroup's waves quantise pieces of 64 * 4 elements of them into aq and asc, which are the launch's own until it ends
    const float* x;
    uint32_t parts, range;           // ranges of K (gridDim.z), steps of each (even)
    float* sums;                     // [workgroup of a range][parts][partial tile]
    uint32_t* arrivals;              // [workgroup of a range], zero between launches
    unsigned long long *flags, id;   // a piece's flag holds the launch's number when the piece is there
    uint32_t spin_limit;
};
constexpr uint32_t FR_PARTS = 4;            // ranges of K at most
constexpr uint32_t FR_PIECES = 2048;         // flags
__host__ __device__ inline uint32_t fr_pieces(uint32_t M, uint32_t K) { return (uint32_t)(((uint64_t)M * K / 4 + 63) / 64); }
__device__ unsigned long long fr_flags[FR_PIECES];

// Piece i of the activations, by one wave.  Other workgroups read it within the launch: stores, and their loads, that say so.
__device__ __forceinline__ void quantise_piece(const FewArgs& a, uint32_t i, uint32_t lane) {
    const uint32_t at = i * 64 + lane, n4 = a.M * a.K / 4;
    const float4 v = at < n4 ? reinterpret_cast<const float4*>(a.x)[at] : make_float4(0.f, 0.f, 0.f, 0.f);
    uint16_t sb;
    const uint32_t packed = quantize_block_part(v, sb, ((at >> 3) % (a.K / 32)) & 1u, true);
    if (at < n4) {
        __hip_atomic_store(reinterpret_cast<uint32_t*>(const_cast<int8_t*>(a.aq)) + at, packed, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if ((at & 7u) == 0) __hip_atomic_store(const_cast<uint16_t*>(a.asc) + (at >> 3), sb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

// One workgroup: 32 MT rows of activations x 32 columns.  SILU: the matrix is [gate; up], a workgroup takes 32 gate columns and the up
// columns of the same indices and writes quantize(silu(gate) * up) as gemm.hip's epilogue does.
// G: groups of 8 rows that are worked out of the last tile of 32 (register r of a tile: rows 8 (r / 4) + 4 h + r % 4); the rest is padding.
// RANGED: a workgroup takes one of a.parts ranges of K.
template <bool Q4, int WAVES, bool SILU, bool BIASED, int MT, int G, bool RAW, bool RANGED>
__global__ __launch_bounds__(WAVES * 64) void gemm_rows_kernel(FewArgs a) {
    constexpr int NT = SILU ? 2 : 1, KW = WAVES / NT;         // column tiles; waves that share K of one
    constexpr int THREADS = WAVES * 64, TILE = 1024 * (MT - 1) + 256 * G;
    constexpr int WB = Q4 ? 64 : 128;                         // bytes of a weight row in a step
    constexpr int LA = MT * 32 * 128, LB = 32 * WB;           // LDS bytes of a step's activation tiles / weight tile
    constexpr int WAVE_LDS = LA + LB;
    static_assert(WAVE_LDS >= TILE * 4, "a wave's strip holds its partial tile");
    __shared__ __attribute__((aligned(16))) uint8_t lds[WAVES * WAVE_LDS];
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t c = lane & 31, h = lane >> 5;
    const uint32_t nblk = a.K / 32, n0 = blockIdx.x * 32, m0 = blockIdx.y * 32 * MT;
    static_assert(!RANGED || (BIASED && !SILU && !RAW && MT == 1), "deep products");
    const uint32_t all = (nblk + FR_U - 1) / FR_U, first = RANGED ? min(all, blockIdx.z * a.range) : 0u, steps = RANGED ? min(all, first + a.range) : all, each = (steps - first + KW - 1) / KW, per = BIASED ? (each + 1) & ~1u : each;
    const uint32_t s0 = min(steps, first + wave % KW * per), s1 = min(steps, s0 + per);
    const uint32_t col0 = n0 + (SILU ? wave / KW * a.inter : 0u);        // this wave's columns: rows col0 .. + 32 of the matrix
    uint8_t* la = lds + wave * WAVE_LDS;                      // this wave's own: no barrier until the partial tiles meet
    uint8_t* lb = la + LA;

    // A wave fetches whole 128-byte (Q4_0: 64-byte) pieces of its rows, eight (four) lanes to a row, and leaves them in its strip of
    // LDS, 16-byte pieces XOR-swizzled by the row; the MFMA operands (one 16-byte piece per lane: row c, half h of a block) come from
    // there.  Fetching the operands directly touches 32 cache lines per instruction, for the scales as well: the vector memory pipe
    // then took longer than the weights' way from memory.  Rows past the end and bytes past the last row read as zero.
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)a.wq, 0, a.N * nblk * (Q4 ? 16 : 32), FR_RSRC);
    const __amdgpu_buffer_rsrc_t rws = __builtin_amdgcn_make_buffer_rsrc((void*)a.wsc, 0, a.N * nblk * 2, FR_RSRC);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)a.aq, 0, a.M * a.K, FR_RSRC);
    const __amdgpu_buffer_rsrc_t ras = __builtin_amdgcn_make_buffer_rsrc((void*)a.asc, 0, a.M * nblk * 2, FR_RSRC);
    constexpr int NLA = 4 * MT, NLB = Q4 ? 2 : 4;                  // loads of a step per tile: 8 rows (Q4_0 weights: 16) each
    const uint32_t ar = lane >> 3, ap = lane & 7;
    const uint32_t br = Q4 ? lane >> 2 : lane >> 3, bp = Q4 ? lane & 3 : lane & 7;
    struct Step { v4i A[NLA], B[NLB]; uint2 sa[MT], sb; };
    // A row's four scales.  An even number of blocks to a row keeps them on 4-byte boundaries and the matrix's end on one; otherwise they
    // are fetched one by one (a word that reaches past the end reads as zero altogether).
    const bool odd_row = (nblk & 1u) != 0;
    auto load_scales = [&](const __amdgpu_buffer_rsrc_t& rsrc, uint32_t at, auto aux) {
        if (!odd_row) return __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rsrc, at, 0, aux.value));
        uint32_t v[FR_U];
#pragma unroll
        for (int u = 0; u < FR_U; u++) v[u] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rsrc, at + 2 * u, 0, aux.value) & 0xFFFFu;
        return make_uint2(v[0] | (v[1] << 16), v[2] | (v[3] << 16));
    };
    auto load_b = [&](Step& g, uint32_t st) {
#pragma unroll
        for (int i = 0; i < NLB; i++)
            g.B[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, (col0 + i * (Q4 ? 16 : 8) + br) * nblk * (Q4 ? 16 : 32) + st * WB + bp * 16, 0, 0);
        g.sb = load_scales(rws, (col0 + c) * nblk * 2 + st * 8, std::integral_constant<int, 0>{});
    };
    auto load_a = [&](Step& g, uint32_t st) {
#pragma unroll
        for (int i = 0; i < NLA; i++) g.A[i] = __builtin_amdgcn_raw_buffer_load_b128(ra, (m0 + i * 8 + ar) * a.K + st * 128 + ap * 16, 0, RAW ? FR_AGENT : 0);
#pragma unroll
        for (int t = 0; t < MT; t++) g.sa[t] = load_scales(ras, (m0 + 32 * t + c) * nblk * 2 + st * 8, std::integral_constant<int, RAW ? FR_AGENT : 0>{});
    };
    auto load = [&](Step& g, uint32_t st) { load_b(g, st); load_a(g, st); };

    float acc[MT][16];
    auto regs = [](int t) { return t < MT - 1 ? 16 : 4 * G; };
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < 16; r++) acc[t][r] = 0.f;
    v16i c_in;
#pragma unroll
    for (int r = 0; r < 16; r++) c_in[r] = BIASED ? (int)FR_MAGIC : 0;
    const v16f zero_f = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    // operand of the rank-1 product: the scale in k = 0 (the lower half-wave's first element), zeros elsewhere
    auto scale_operand = [&](uint32_t bits) {
        const _Float16 z = (_Float16)0.0f;
        return (v4h){__builtin_bit_cast(_Float16, (uint16_t)(h ? 0u : bits)), z, z, z};
    };
    auto scale_of = [](const uint2& v, int u) { return (u < 2 ? v.x : v.y) >> (16 * (u & 1)); };
    // the scales of a step as they count: 0 past the end of K (those are the next row's), a minus sign on the weights' odd blocks
    auto valid_scales = [&](uint2 v, uint32_t st, bool weights) {
        const uint32_t left = st * FR_U < nblk ? nblk - st * FR_U : 0u;
        v.x = left > 1 ? v.x : left ? v.x & 0xFFFFu : 0u;
        v.y = left > 3 ? v.y : left > 2 ? v.y & 0xFFFFu : 0u;
        if (weights) { v.x ^= 0x80000000u; v.y ^= 0x80000000u; }
        return v;
    };

    auto compute = [&](Step& g, uint32_t st) {
#pragma unroll
        for (int t = 0; t < MT; t++) g.sa[t] = valid_scales(g.sa[t], st, false);
        g.sb = valid_scales(g.sb, st, true);
#pragma unroll
        for (int i = 0; i < NLA; i++) {
            const uint32_t row = i * 8 + ar;
            *reinterpret_cast<v4i*>(la + row * 128 + ((ap ^ ((row >> 1) & 7)) * 16)) = g.A[i];
        }
#pragma unroll
        for (int i = 0; i < NLB; i++) {
            const uint32_t row = i * (Q4 ? 16 : 8) + br;
            *reinterpret_cast<v4i*>(lb + row * WB + ((bp ^ (Q4 ? (row >> 2) & 3 : (row >> 1) & 7)) * 16)) = g.B[i];
        }
#pragma unroll
        for (int u = 0; u < FR_U; u++) {
            v4i B;
            if (Q4) {
                const v4i p = *reinterpret_cast<const v4i*>(lb + c * WB + ((u ^ ((c >> 2) & 3)) * 16));
                // elements 0..15 in the low nibbles, 16..31 in the high ones, as 16 (code - 8): the sum is divided by 16 at the end
                const uint32_t sh = h ? 0u : 4u;
#pragma unroll
                for (int i = 0; i < 4; i++) B[i] = (int)((((uint32_t)p[i] << sh) & 0xF0F0F0F0u) ^ 0x80808080u);
            } else {
                B = *reinterpret_cast<const v4i*>(lb + c * WB + (((2 * u + h) ^ ((c >> 1) & 7)) * 16));
            }
            const v4h fb = scale_operand(scale_of(g.sb, u));
#pragma unroll
            for (int t = 0; t < MT; t++) {
                const v4i A = *reinterpret_cast<const v4i*>(la + (32 * t + c) * 128 + (((2 * u + h) ^ ((c >> 1) & 7)) * 16));
                const v16i isum = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B, c_in, 0, 0, 0);
                const v16f S = __builtin_amdgcn_mfma_f32_32x32x8f16(scale_operand(scale_of(g.sa[t], u)), fb, zero_f, 0, 0, 0);
                const v16f biased = __builtin_bit_cast(v16f, isum);          // 12582912 +- block sum
#pragma unroll
                for (int r = 0; r < regs(t); r++) acc[t][r] = fmaf(S[r], BIASED ? biased[r] : (float)isum[r], acc[t][r]);
            }
        }
        // the sums are final here: left alone, the compiler works on two steps' products at once and has no registers for them
#pragma unroll
        for (int t = 0; t < MT; t++)
#pragma unroll
            for (int r = 0; r < regs(t); r++) asm volatile("" : "+v"(acc[t][r]));
    };
    // What eight blocks left of the bias, 1.5 * 2^23 * sum_b a_s[b] * (+-w_s[b]), off the sums: gemm.hip's f16 MFMA over the same eight
    // blocks (most of the biased sums' rounding is made here, and the same eight blocks make the same).
    auto unbias = [&](const uint2 (&a0)[MT], const uint2 (&a1)[MT], uint2 w0, uint2 w1) {
        const _Float16 af = (_Float16)(float)(1 << FR_A_LOG2);
        const _Float16 bf = h ? (_Float16)(-(float)(1 << (22 - FR_A_LOG2))) : (_Float16)(-(float)(1 << (23 - FR_A_LOG2)));
        const v8h tb = __builtin_bit_cast(v8h, make_uint4(w0.x, w0.y, w1.x, w1.y)) * (v8h){bf, bf, bf, bf, bf, bf, bf, bf};
#pragma unroll
        for (int t = 0; t < MT; t++) {
            const v8h ta = __builtin_bit_cast(v8h, make_uint4(a0[t].x, a0[t].y, a1[t].x, a1[t].y)) * (v8h){af, af, af, af, af, af, af, af};
            v16f d;
#pragma unroll
            for (int r = 0; r < 16; r++) d[r] = acc[t][r];
            d = __builtin_amdgcn_mfma_f32_32x32x16_f16(ta, tb, d, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 16; r++) acc[t][r] = d[r];
        }
    };
    // two steps in flight
    Step x0, x1;
    if constexpr (RAW) {
        // A wave's pieces first, then its weights, which are on their way while everybody's pieces are waited for.
        const uint32_t n = fr_pieces(a.M, a.K), grid = gridDim.x * gridDim.y;
        __shared__ uint32_t late;
        if (tid == 0) late = 0;
        for (uint32_t i = blockIdx.y * gridDim.x + blockIdx.x + wave * grid; i < n; i += WAVES * grid) {
            quantise_piece(a, i, lane);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");         // acknowledged
            if (lane == 0) __hip_atomic_store(a.flags + i, a.id, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (s0 < s1) load_b(x0, s0);
        if (s0 + 1 < s1) load_b(x1, s0 + 1);
        __syncthreads();
        for (uint32_t p = tid; p < n; p += THREADS) {
            uint32_t rounds = 0;
            while (__hip_atomic_load(a.flags + p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != a.id)
                if (++rounds >= a.spin_limit) { late = 1; break; }
        }
        __syncthreads();
        if (late) {                                                  // somebody is not there: the same codes once more
            for (uint32_t j = wave; j < n; j += WAVES) quantise_piece(a, j, lane);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            __syncthreads();
        }
        if (s0 < s1) load_a(x0, s0);
        if (s0 + 1 < s1) load_a(x1, s0 + 1);
    } else {
        if (s0 < s1) load(x0, s0);
        if (s0 + 1 < s1) load(x1, s0 + 1);
    }
    for (uint32_t st = s0; st < s1; st += 2) {
        compute(x0, st);
        uint2 a0[MT], a1[MT], w0 = x0.sb, w1 = make_uint2(0u, 0u);
#pragma unroll
        for (int t = 0; t < MT; t++) { a0[t] = x0.sa[t]; a1[t] = w1; }
        if (st + 2 < s1) load(x0, st + 2);
        if (st + 1 < s1) {
            compute(x1, st + 1);
#pragma unroll
            for (int t = 0; t < MT; t++) a1[t] = x1.sa[t];
            w1 = x1.sb;
        }
        if (st + 3 < s1) load(x1, st + 3);
        if (BIASED) unbias(a0, a1, w0, w1);
    }

    // lane: column c, rows 8 (r / 4) + 4 h + r % 4 of a tile of 32.  Element e = (16 t + r) * 64 + lane of a partial tile; the waves' partial tiles are
    // added in the order of K.
    float* red = reinterpret_cast<float*>(la);
#pragma unroll
    for (int t = 0; t < MT; t++)
#pragma unroll
        for (int r = 0; r < regs(t); r++) red[(16 * t + r) * 64 + lane] = acc[t][r];
    __syncthreads();
    const uint32_t group = RANGED ? blockIdx.y * gridDim.x + blockIdx.x : 0u;
    float* mine = RANGED ? a.sums + (size_t)group * a.parts * TILE : nullptr;
    if constexpr (RANGED) {
        // The ranges' partial tiles meet in memory, past the caches of an XCD.  A wave's stores have arrived before the barrier that lets the workgroup count itself in; who
        // counts `parts` adds them up in the order of K and leaves the counter at zero.
        for (uint32_t e = tid; e < TILE; e += THREADS) {
            float p[KW];
#pragma unroll
            for (int w = 0; w < KW; w++) p[w] = reinterpret_cast<const float*>(lds + w * WAVE_LDS)[e];
#pragma unroll
            for (int w = 1; w < KW; w++) p[0] = p[0] + p[w];
            __hip_atomic_store(mine + (size_t)blockIdx.z * TILE + e, p[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __shared__ uint32_t arrived;
        __syncthreads();
        if (tid == 0) {
            arrived = __hip_atomic_fetch_add(a.arrivals + group, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
            if (arrived == a.parts) __hip_atomic_store(a.arrivals + group, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        __syncthreads();
        if (arrived != a.parts) return;
    }
    for (uint32_t e = tid; e < TILE; e += THREADS) {
        float v[NT];
        if constexpr (RANGED) {
            float p[FR_PARTS];
#pragma unroll
            for (uint32_t q = 0; q < FR_PARTS; q++) p[q] = __hip_atomic_load(mine + (size_t)min(q, a.parts - 1) * TILE + e, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            v[0] = p[0];
#pragma unroll
            for (uint32_t q = 1; q < FR_PARTS; q++) v[0] = q < a.parts ? v[0] + p[q] : v[0];
            if (Q4) v[0] *= 0.0625f;
        } else
#pragma unroll
        for (int j = 0; j < NT; j++) {
            float p[KW];
#pragma unroll
            for (int w = 0; w < KW; w++) p[w] = reinterpret_cast<const float*>(lds + (j * KW + w) * WAVE_LDS)[e];
            v[j] = p[0];
#pragma unroll
            for (int w = 1; w < KW; w++) v[j] = v[j] + p[w];
            if (Q4) v[j] *= 0.0625f;
        }
        const uint32_t r = e >> 6, el = e & 63, col = el & 31;
        const uint32_t m = m0 + 8 * (r >> 2) + 4 * (el >> 5) + (r & 3);       // (32 rows further on every 16 r)
        if (SILU) {
            // gemm.hip's epilogue: the 32 lanes of a half-wave are one block of one row
            const float o = v[0] * __builtin_amdgcn_rcpf(1.0f + __expf(-v[0])) * v[NT - 1];
            const float amax = half_wave_max(fabsf(o));
            const float scl = amax * (1.0f / 127.0f);
            float inv = amax > 0.f ? 127.0f * __builtin_amdgcn_rcpf(amax) : 0.f;
            if (blockIdx.x & 1u) inv = -inv;
            const uint32_t code = (uint32_t)(int)__builtin_rintf(o * inv) & 0xFFu;
            const uint32_t pk = quad_broadcast<0>(code) | (quad_broadcast<1>(code) << 8) | (quad_broadcast<2>(code) << 16) | (quad_broadcast<3>(code) << 24);
            if (m < a.M) {
                if ((col & 3u) == 0) *reinterpret_cast<uint32_t*>(a.silu_q + (size_t)m * a.inter + n0 + col) = pk;
                if (col == 0) a.silu_sc[(size_t)m * (a.inter / 32) + blockIdx.x] = f32_to_f16_bits(scl);
            }
        } else if (m < a.M && n0 + col < a.N) {
            float* dst = a.y + (size_t)m * a.ldy + n0 + col;
            *dst = a.accumulate ? *dst + v[0] : v[0];
        }
    }
}

template <bool Q4, bool SILU, int MT, int G, bool RAW>
void launch_groups(const FewArgs& a, hipStream_t s) {
    constexpr int WAVES = 8;       // sixteen leave a wave 128 registers, and two steps in flight do not fit them
    const dim3 grid(((SILU ? a.inter : a.N) + 31) / 32, (a.M + 32 * MT - 1) / (32 * MT), a.parts);
    if constexpr (!SILU && !RAW && MT == 1)
        if (a.parts > 1) { fh::launch(gemm_rows_kernel<Q4, WAVES, SILU, true, MT, G, RAW, true>, grid, WAVES * 64, 0, s, a); return; }
    if (a.K > 4096) fh::launch(gemm_rows_kernel<Q4, WAVES, SILU, true, MT, G, RAW, false>, grid, WAVES * 64, 0, s, a);
    else fh::launch(gemm_rows_kernel<Q4, WAVES, SILU, false, MT, G, RAW, false>, grid, WAVES * 64, 0, s, a);
}
template <bool Q4, bool SILU, int MT, bool RAW>
void launch_rows(const FewArgs& a, hipStream_t s) {
    // one row of workgroups: its last tile's rows are known here
    const uint32_t left = a.M > 32 * (MT - 1) && a.M <= 32 * MT ? a.M - 32 * (MT - 1) : 32;
    if (left <= 8) launch_groups<Q4, SILU, MT, 1, RAW>(a, s);
    else if (left <= 16) launch_groups<Q4, SILU, MT, 2, RAW>(a, s);
    else launch_groups<Q4, SILU, MT, 4, RAW>(a, s);
}

}  // namespace

static unsigned long long* fr_flags_of_device() {
    constexpr int MAX = 16;
    static std::atomic<unsigned long long*> of[MAX] = {};
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= MAX) return nullptr;
    unsigned long long* p = of[dev].load(std::memory_order_relaxed);
    if (!p) {
        void* v = nullptr;
        if (hipGetSymbolAddress(&v, HIP_SYMBOL(fr_flags)) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
        of[dev].store(p = static_cast<unsigned long long*>(v), std::memory_order_relaxed);
    }
    return p;
}

// 32-bit byte offsets, and a grid's second dimension ends at 65535 (2.1 million rows, which its estimate would take for narrow, shallow matrices).
bool gemm_rows_supported(const QWeight& w, uint32_t M, bool silu) {
    return (!silu || w.N % 64 == 0) && M <= 65535u * 32u && (uint64_t)M * w.K <= 0x7FFFFFFFull && (uint64_t)w.N * std::max<uint64_t>(w.qs_row_bytes(), w.K / 16) <= 0x7FFFFFFFull;
}

// Ranges of K, one to a workgroup, for deep products whose tiles leave half the compute units idle: a workgroup takes 20 bytes of weights a nanosecond, and 64 of them 14 us for
// 8192 -> 2048.  us with the quantiser, whole / in ranges (six operand sets in turn): Q8_0 8192 -> 2048 by 5 rows 15.1 / 11.8, 32 (4 ranges) 16.1 / 11.9, 64 (2) 16.3 / 13.7, 8192 -> 3072
// by 16 15.3 / 12.2, Q4_0 8192 -> 2048 by 32 14.8 / 12.0.  Not two ranges with two rows of tiles to a workgroup (8192 -> 2048 by 100 16.3 / 18.6).
// Shallower ones, whole (the quantiser in the launch where that pays) / in ranges, by 5, 16, 32 and 64 rows: Q8_0 4096 -> 1024 8.1 / 11.1, 9.1 / 11.1, 10.4 / 11.2, 10.5 / 11.0, 5632 -> 2048 10.2 / 10.9,
// 11.4 / 10.9, 12.5 / 10.9, 12.7 / 12.0, 7168 -> 2048 12.0 / 10.9, 13.4 / 10.9, 15.0 / 11.5, 15.0 / 13.1; Q4_0 4096 -> 2048 8.4 / 11.2, 8.8 / 11.1, 10.5 / 11.2, 10.7 / 11.0, 5632 -> 2048 10.0 / 11.0,
// 11.2 / 11.0, 11.8 / 11.0, 12.1 / 12.0, 7168 -> 2048 11.5 / 11.0, 12.6 / 11.0, 13.9 / 11.3, 14.2 / 12.8.  The two meet about 5632; the line is at 8192, the depth of the first measurements, and
// gives away 1 to 3 us from there on.
static uint32_t ranges(const QWeight& w, uint32_t M) {
    const uint64_t grid = (uint64_t)((w.N + 31) / 32) * ((M + 31) / 32);
    return w.K >= 8192 && M <= 64 && grid <= 128 ? (uint32_t)std::min<uint64_t>(FR_PARTS, 256 / grid) : 1;
}

// Rounds of 256 tiles of 32 columns by 32 `mt` rows, one to a compute unit (a SiLU workgroup works two columns of them).
static uint32_t rounds(const QWeight& w, uint32_t M, uint32_t mt) { return (uint32_t)(((uint64_t)((w.N + 31) / 32) * ((M + 32 * mt - 1) / (32 * mt)) + 255) / 256); }

// Rows of tiles to a workgroup.  Two share the weights, their way through LDS and the nibbles' arithmetic: a round takes 1.6 times as long
// (1.4 to 1.7; 1.8 where the sums are biased), so they pay where they save more than that in rounds.  us with the quantiser, one row of tiles / two, Q4_0: 2048 -> 8192 by 33
// rows 12.4 / 10.6, 64 13.1 / 11.4, 65 (3 rounds against 2) 17.2 / 17.6, 100 21.9 / 18.5; 8192 -> 2048 by 128 17.4 / 22.6, by 256 31.5 / 27.1; 3072 -> 1024
// by 300 15.5 / 13.9.  The same bits either way.
static double two_rows_take(const QWeight& w) { return w.K > 4096 ? 1.8 : 1.6; }
static uint32_t tile_rows(const QWeight& w, uint32_t M) {
    return two_rows_take(w) * rounds(w, M, 2) < rounds(w, M, 1) ? 2 : 1;
}

// Whether one launch quantises the activations too.  The hand-over of the codes inside it (2 us) hides where a caller's loop waits for the host's launches (9.6 us for two, 6.5 for
// one), or where they are few.  us, two launches / one, Q4_0: 576 -> 1536 by 2 .. 200 rows 9.7 / 7.4, 2048 -> 2048 by 2 .. 64 9.5 / 7.3, by 128 9.5 / 8.1, 2048 -> 512 by 16 9.6 / 7.4,
// 128 (two pieces a wave) 9.7 / 9.1, 2048 -> 8192 by 2 9.7 / 7.8, 32 9.6 / 8.7, 64 (two tiles) 11.2 / 11.2, 8192 -> 2048 by 8 13.4 / 12.0, 32 14.4 / 15.3, 3072 -> 8192 by 2 9.6 / 9.2,
// 16 9.9 / 10.8, 3072 -> 1024 by 16 9.4 / 7.4, 64 9.4 / 9.5; Q8_0 2048 -> 8192 by 16 9.8 / 9.4, 32 9.5 / 9.7.
// The whole grid has to be at work at a time (512 workgroups: those at work wait until they give up).  Recorded into a graph the launch would find its number from the replay before.
bool gemm_rows_raw(const QWeight& w, uint32_t M, bool ranged, hipStream_t s) {
    if (ranged && ranges(w, M) > 1) return false;      // 8192 -> 2048 by 2 to 8 rows, one launch / ranges: Q8_0 13.1 / 11.9, Q4_0 12.2 / 11.7
    const uint64_t grid = (w.N + 31) / 32 * (((uint64_t)M + 31) / 32), bytes = (uint64_t)w.N * w.qs_row_bytes();
    const bool pays = M <= 8 ? bytes <= (20u << 20) : M <= 16 ? w.K <= 2048 || bytes <= (4u << 20) : w.K <= 2048 && bytes <= (10u << 20);
    hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
    return pays && tile_rows(w, M) == 1 && grid <= 256 && fr_pieces(M, w.K) <= std::min<uint64_t>(FR_PIECES, 16 * grid) && fr_flags_of_device() &&
           hipStreamIsCapturing(s, &st) == hipSuccess && st == hipStreamCaptureStatusNone;
}

// Microseconds of a launch, for the choice between the kernels.  Tiles come in rounds of one to a compute unit; a round takes 1.8 plus 2.7 per
// 2048 of depth, or what its columns take from memory at 4.8 TB/s (with the quantiser, 1 / 2 / 3 / 4 rounds: K = 2048 9.9 / 14.2 / 18.8 / 23.5,
// K = 4096 13 / 20 / 27 / 34, K = 8192 17.5 / 29 / 40 / 52).  1422 products of 2 to 1300 rows were timed both ways, with one row of tiles to a
// workgroup: the kernel that the estimates prefer is within 3 % of the faster one in all but 9, within 8 % in all.
double gemm_rows_cost(const QWeight& w, uint32_t M, bool ranged) {
    const uint32_t mt = tile_rows(w, M), parts = ranged && mt == 1 ? ranges(w, M) : 1;
    if (parts > 1) return 6.0 + 2.7 * w.K / 2048.0 / parts;
    const double columns = std::min<uint32_t>(w.N, 256 * 32), row_bytes = (double)w.qs_row_bytes() + w.K / 16;
    return 2.0 + (double)rounds(w, M, mt) * std::max((mt == 2 ? two_rows_take(w) : 1.0) * (1.8 + 2.7 * w.K / 2048.0), columns * row_bytes / 4.8e6);
}

void launch_gemm_rows(const QWeight& w, const int8_t* aq, const uint16_t* as, uint32_t M, float* y, uint32_t ldy, bool accumulate, hipStream_t s,
                      int8_t* silu_q, uint16_t* silu_sc, const float* raw, const GemmRowsSums* sums) {
    const bool ranged = sums && !silu_q && !raw;
    const uint32_t mt = raw ? 1 : tile_rows(w, M);
    FewArgs a{w.qs, w.scales, aq, as, y, M, w.N, w.K, ldy, accumulate ? 1u : 0u, silu_q, silu_sc, w.N / 2, raw, 1, 0, nullptr, nullptr, nullptr, 0, 0};
    const uint32_t steps = (w.K / 32 + FR_U - 1) / FR_U;
    if (ranged && mt == 1 && ranges(w, M) > 1) { a.parts = ranges(w, M); a.sums = sums->partials; a.arrivals = sums->counters; }
    a.range = ((steps + a.parts - 1) / a.parts + 1) & ~1u;
    if (raw) {
        static const uint32_t limit = [] { const char* e = getenv("FORGE_HIP_PD_SPIN_LIMIT"); return e && atoi(e) > 0 ? (uint32_t)atoi(e) : 64u; }();
        a.spin_limit = limit;
        static std::atomic<unsigned long long> number{0};
        a.id = ++number;
        a.flags = fr_flags_of_device();
    }
    const bool q4 = w.wdtype == FORGE_HIP_Q4_0, silu = silu_q != nullptr;
    auto go = [&](auto q4_, auto silu_) {
        if (mt == 2) launch_rows<decltype(q4_)::value, decltype(silu_)::value, 2, false>(a, s);
        else launch_rows<decltype(q4_)::value, decltype(silu_)::value, 1, false>(a, s);
    };
    if (raw && q4) launch_rows<true, false, 1, true>(a, s);
    else if (raw) launch_rows<false, false, 1, true>(a, s);
    else if (q4 && silu) go(std::true_type{}, std::true_type{});
    else if (q4) go(std::true_type{}, std::false_type{});
    else if (silu) go(std::false_type{}, std::true_type{});
    else go(std::false_type{}, std::false_type{});
}

}  // namespace fh
