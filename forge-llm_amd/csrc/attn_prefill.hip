// Batched-prefill causal attention (attention_flash_batch, emit.rs:754-883) over an fp16 KV
// cache, with both matrix products on fp16 MFMA (v_mfma_f32_32x32x16_f16) and the online
// softmax in f32.
//
// Workgroup = 128 consecutive queries of one head in four groups of 32; four waves, one to a group, or eight, two to a group, which take one
// half (32 keys) of every key tile and merge their (max, sum, output) once at the end, so that the longest chain of dependent tile steps
// (the last query tile's) is worked on by twice the waves.
// K/V are streamed in tiles of 64 keys through two LDS buffers, both as rows, by loads that go straight into LDS: no registers, one offset per
// lane that every tile reuses behind a new descriptor, one wait and one barrier per step.  P.V wants V with the keys contiguous per lane:
// ds_read_b64_tr_b16 transposes on the way out.  (Through registers, with V transposed on the way in, a third of a step went into issuing the
// loads and writing them to LDS, and the registers they took left two waves per SIMD where three fit now.)
// Scores stay in the base-2 domain (s * scale * log2 e) so that the exponential is one v_exp_f32 after one FMA; keys are masked only in
// tiles that reach past the wave's first query; accumulators are rescaled only when some query's maximum rises.  (Letting a maximum stand until a score passes
// it by 2^8 saves 3 of 80 us at 3001 tokens, but the largest weight is then no longer exactly 1 in fp16: error against 64 bits 2.45e-4 instead of 2.35e-4.  Not kept.)
// What bounds it: full, 768 cycles of the matrix unit and about 860 of the VALU (32 exp, 32 FMA, 32 additions, 16 conversions, 16 maxima per 32 x 64 scores, heads of 96), hardly
// any of them beside one another, in about 1620; LDS is busy a third of the time, of 128 nearly half (heads of 96, 3072 queries behind 8192 keys 410 us = 0.89 PFLOP/s, 128 0.93, 64
// 0.80; the library's large bf16 product is at 1.2); causal, the uneven length of the query tiles on top.  3001 tokens: 32/32 heads of 96 97.7 -> 80 us,
// 32/8 of 128 124 -> 96, 2502 tokens of 32/8 of 64 52.5 -> 46.9, 1000 of 32/8 of 128 38.2 -> 28.
// Measured and not kept: query tiles of every other round in ascending order: within 2 %.
//
// Both products are computed transposed, S^T = K Q^T and O^T = V^T P^T.  In the 32x32 MFMA
// result layout a lane then owns ONE query (column = lane%32) and 16 keys (or 16 head dims),
// so the softmax row statistics are per-lane scalars (plus one exchange with lane^32), and
// the exponentiated scores are already in the register layout the second MFMA wants for
// its B operand.
#include "common.h"
#include "device_utils.h"

namespace fh {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));
typedef short v4s __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));

constexpr int QW = 32;        // queries per wave pair
constexpr int QB = 128;       // queries per workgroup
constexpr int KT = 64;        // keys per tile
constexpr int AP_THREADS = 512;   // the 8-wave form; the 4-wave form runs 256
constexpr uint32_t AP_RSRC_FLAGS = 0x00020000;   // raw buffer, 32-bit data format

#define FH_LDS3(p) ((__attribute__((address_space(3))) void*)(p))

// Where piece p (16 bytes) of row r of a tile lies in its row of LDS, and which piece lies at p: eight consecutive rows of K at one piece
// (a fragment's reads), and two neighbouring pieces of four consecutive rows of V, touch 128 bytes' worth of banks once.  By the counters that is half of what LDS serves at once: a third (heads of
// 64 and 96) to a half (128) of its active cycles are conflicts, of a unit that is busy 29 to 44 % of the time.  Rows are as long in LDS as they are: a load
// into LDS fills 1 KB in lane order.
template <int HD>
__device__ __forceinline__ uint32_t piece_of(uint32_t r, uint32_t p) {
    if constexpr (HD == 96) return p ^ ((r & 2) | ((r >> 2) & 1));       // rows alternate between two halves of the banks as they are
    else return p ^ (((r & 3) << 1) | ((r >> 2) & 1));
}

__device__ __forceinline__ v4h read_transposed(const uint8_t* at) {
    return __builtin_bit_cast(v4h, __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) v4s*)at));
}

// The compiler waits for everything that is on its way into LDS ahead of a transposing read of its own, that is for the next tiles in the middle of a step; reads in
// assembly have waits of their own, which keep them from running ahead of the products.  What is the better differs by form and head, hardly by whether heads share K and V.
// us, the compiler's waits / own, 32/32 and 32/8 heads:
//   eight waves, 1000 rows         64 21.3 / 20.5, 20.1 / 19.3    96 24.4 / 23.5, 24.6 / 23.4    128 27.1 / 27.9, 26.9 / 27.7
//   1024 behind 4096               64 76.0 / 70.8, 73.6 / 68.7    96 111.8 / 96.0, 90.8 / 85.1    128 113.8 / 106.2, 102.1 / 105.2
//   four waves, 3001               64 68.3 / 69.2, 58.2 / 58.5    96 85.4 / 84.7, 77.6 / 77.3    128 100.1 / 102.4, 93.9 / 95.9
//   2048 behind 8192               64 209.9 / 217.3, 202.7 / 208.3    96 283.9 / 279.7, 277.4 / 278.9    128 340.4 / 346.3, 334.1 / 342.6
template <int HD, int KH> constexpr bool own_waits() { return HD == 96 || (HD == 64 && KH == 1); }

// V fragments of 32 keys: f[j][d] = keys 16 j + 4 lh .. + 3 and + 8 of dim 32 d + lane % 32.  at0, at1: LDS addresses of this lane's part of the first dims and of those 32 further on
// (a row's swizzle is the same again 64 further; with heads of 96 it is the same everywhere).
#define FH_TR(dst, at, off) "ds_read_b64_tr_b16 " dst ", " at " offset:" off "\n"
#define FH_TR4(a, b, c, d, at, off) FH_TR(a, at, off) FH_TR(b, at, off "+%[k8]") FH_TR(c, at, off "+%[k8]*2") FH_TR(d, at, off "+%[k8]*3")
template <int HD>
__device__ __forceinline__ void read_v(v8h (&f)[2][HD / 32], uint32_t at0, uint32_t at1) {
    v4h r[3][4];
    if constexpr (HD == 96)
        asm volatile(FH_TR4("%[x00]", "%[x01]", "%[x02]", "%[x03]", "%[at0]", "0") FH_TR4("%[x10]", "%[x11]", "%[x12]", "%[x13]", "%[at0]", "64")
                     FH_TR4("%[x20]", "%[x21]", "%[x22]", "%[x23]", "%[at0]", "128") "s_waitcnt lgkmcnt(0)"
                     : [x00] "=&v"(r[0][0]), [x01] "=&v"(r[0][1]), [x02] "=&v"(r[0][2]), [x03] "=&v"(r[0][3]), [x10] "=&v"(r[1][0]), [x11] "=&v"(r[1][1]),
                       [x12] "=&v"(r[1][2]), [x13] "=&v"(r[1][3]), [x20] "=&v"(r[2][0]), [x21] "=&v"(r[2][1]), [x22] "=&v"(r[2][2]), [x23] "=&v"(r[2][3])
                     : [at0] "v"(at0), [k8] "n"(8 * 2 * HD));
    else
        asm volatile(FH_TR4("%[x00]", "%[x01]", "%[x02]", "%[x03]", "%[at0]", "0") FH_TR4("%[x10]", "%[x11]", "%[x12]", "%[x13]", "%[at1]", "0") "s_waitcnt lgkmcnt(0)"
                     : [x00] "=&v"(r[0][0]), [x01] "=&v"(r[0][1]), [x02] "=&v"(r[0][2]), [x03] "=&v"(r[0][3]), [x10] "=&v"(r[1][0]), [x11] "=&v"(r[1][1]),
                       [x12] "=&v"(r[1][2]), [x13] "=&v"(r[1][3])
                     : [at0] "v"(at0), [at1] "v"(at1), [k8] "n"(8 * 2 * HD));
#pragma unroll
    for (int d = 0; d < HD / 32; d++)
#pragma unroll
        for (int j = 0; j < 2; j++) f[j][d] = __builtin_shufflevector(r[d][2 * j], r[d][2 * j + 1], 0, 1, 2, 3, 4, 5, 6, 7);
}
#undef FH_TR4
#undef FH_TR

// QUANT: instead of f32 rows the kernel writes what the o projection's GEMM reads, the activation quantiser's int8
// codes oq[M][heads*HD] and fp16 scales osc[M][heads*HD/32] of the same values (a 32-element block is one 32-wide
// head_dim tile of one query: 16 values in this lane, 16 in lane ^ 32).
// WIN: sliding-window attention (attention_sliding_batch, emit.rs:907-1046): the query at position p sees the keys
// [max(0, p - window + 1), p]; key tiles that lie before the window of the workgroup's first query are never loaded.
// KH: 32-key halves of a tile that one wave works.  1 = the 8-wave form described above (two waves share a query group and
// merge at the end: twice the waves on the longest chain, for short sequences); 2 = 4 waves, each takes its 32 queries
// through all 64 keys of a tile: two independent score tiles per step to overlap, one maximum / rescale / lane exchange
// per 64 keys, no merge.
// DIRECT: tiles go straight into LDS, whose loads want the cache on a 16-byte boundary.  Otherwise through registers, in the same places: a cache may begin anywhere.
template <int HD, bool QUANT, bool WIN, int KH, bool DIRECT>
__global__ __launch_bounds__(AP_THREADS / KH) __attribute__((amdgpu_waves_per_eu(2)))
void attn_prefill_kernel(const float* __restrict__ q, const uint16_t* __restrict__ kc_flat, const uint16_t* __restrict__ vc_flat,
                         float* __restrict__ out, uint32_t q_stride, uint32_t out_stride, uint32_t M, uint32_t base_pos,
                         uint32_t heads, uint32_t kv_heads, int8_t* __restrict__ oq, uint16_t* __restrict__ osc, uint32_t window,
                         PageTable pt) {
    constexpr uint32_t ROW = HD * 2, PIECES = HD / 8;     // bytes and 16-byte pieces of a row of a tile
    constexpr uint32_t TILE = KT * ROW;                   // bytes of a tile of K, and of V
    constexpr uint32_t WAVES = AP_THREADS / KH / 64;
    constexpr uint32_t LOADS = 2 * PIECES / WAVES;        // loads of 1 KB into LDS per wave and tile pair: K's come first
    constexpr bool EVEN = PIECES % WAVES == 0;            // then a wave's loads of V repeat those of K
    constexpr uint32_t OFFS = EVEN ? LOADS / 2 : LOADS;
    constexpr bool OWN = own_waits<HD, KH>();
    constexpr int NS = HD / 16;   // MFMA k-steps over head_dim
    constexpr int ND = HD / 32;   // 32-wide head_dim tiles of the output
    constexpr int MERGE_FLOATS = 2 + ND * 16;    // per lane: m, l and the output accumulators
    // two pairs of tiles: those of step t+1 arrive while the ones of step t are read, one barrier per step
    constexpr uint32_t LDS = KH == 1 && 4 * 64 * MERGE_FLOATS * 4 > 4 * TILE ? 4 * 64 * MERGE_FLOATS * 4 : 4 * TILE;
    __shared__ __attribute__((aligned(16))) uint8_t smem[LDS];

    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t qg = KH == 1 ? wave >> 1 : wave, kh = KH == 1 ? (wave & 1) : 0;   // query group of 32, (first) half of every key tile
    const uint32_t lq = lane & 31, lh = lane >> 5;
    // tile-major order, heaviest (latest) query tiles first: they stream the most keys, and whatever does not fit the
    // machine at once is the light end, handed out as the first workgroups finish
    const uint32_t head = blockIdx.x % heads, kvh = head / (heads / kv_heads);
    const uint32_t ntq = gridDim.x / heads;
    const uint32_t qtile = ntq - 1 - blockIdx.x / heads;
    const uint32_t q0 = qtile * QB;
    const uint32_t kv_stride = kv_heads * HD;
    const uint32_t seq_total = base_pos + M;
    // scores are kept in the base-2 domain: s * (scale * log2 e), so that exp is the bare v_exp_f32
    const float c2 = (1.0f / sqrtf((float)HD)) * 1.4426950408889634f;

    const uint32_t qrow = q0 + qg * QW + lq;
    const uint32_t qpos = base_pos + qrow;
    v16f oacc[ND];
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[d][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    const uint32_t wg_max_pos = base_pos + min(q0 + QB, M) - 1;
    const uint32_t ntiles = wg_max_pos / KT + 1;
    const uint32_t wave_max_pos = base_pos + min(q0 + qg * QW + QW, M) - 1;   // may underflow if the group is empty
    const uint32_t wave_min_pos = base_pos + q0 + qg * QW;                    // position of the group's first query
    const bool wave_active = q0 + qg * QW < M;
    // first key any query of the workgroup / of this wave's group may see
    const uint32_t wg_lo = (WIN && base_pos + q0 + 1 > window) ? base_pos + q0 + 1 - window : 0;
    const uint32_t wave_lo = (WIN && wave_min_pos + 1 > window) ? wave_min_pos + 1 - window : 0;
    const uint32_t tile0 = wg_lo / KT;

    // Load j of a step (a wave's are wave, wave + WAVES, ...) fills 1 KB of K (j < PIECES) or V, lane -> 16-byte piece; which piece of its row
    // that is follows from the swizzle.  Rows past the last key read 0.
    uint32_t off[OFFS];
#pragma unroll
    for (uint32_t i = 0; i < OFFS; i++) {
        const uint32_t p = (wave + WAVES * i) % PIECES * 64 + lane, row = p / PIECES;
        off[i] = row * kv_stride * 2 + piece_of<HD>(row, p % PIECES) * 16;
    }
    uint4 held[DIRECT ? 1 : LOADS];
    auto load_tiles = [&](uint32_t kt, uint32_t buf) {
        // a paged cache: a tile of 64 keys lies within one page (pages are multiples of 64 rows)
        const size_t at = paged_row(pt, kt * KT) * kv_stride + kvh * HD;
        const uint32_t records = (uint32_t)__builtin_amdgcn_readfirstlane((int)((min(seq_total - kt * KT, (uint32_t)KT) - 1) * kv_stride * 2 + ROW));
        if constexpr (DIRECT) {
#pragma unroll
            for (uint32_t i = 0; i < LOADS; i++) {
                const uint32_t j = wave + WAVES * i;
                const bool of_k = EVEN ? i < PIECES / WAVES : j < PIECES;
                const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)((of_k ? kc_flat : vc_flat) + at), 0, records, AP_RSRC_FLAGS);
                const uint32_t at_lane = off[i % OFFS];
                __builtin_amdgcn_raw_ptr_buffer_load_lds(r, FH_LDS3(smem + buf * 2 * TILE + j * 1024), 16, at_lane, 0, 0, 0);
            }
        } else {
#pragma unroll
            for (uint32_t i = 0; i < LOADS; i++) {
                const uint32_t j = wave + WAVES * i, at_lane = off[i % OFFS];
                held[i] = make_uint4(0u, 0u, 0u, 0u);
                if (at_lane < records) __builtin_memcpy(&held[i], reinterpret_cast<const uint8_t*>((j < PIECES ? kc_flat : vc_flat) + at) + at_lane, 16);
            }
        }
    };
    auto put_tiles = [&](uint32_t buf) {
#pragma unroll
        for (uint32_t i = 0; i < LOADS; i++) *reinterpret_cast<uint4*>(smem + buf * 2 * TILE + (wave + WAVES * i) * 1024 + lane * 16) = held[i];
    };
    // Addresses of the fragments in LDS.  K (A operand): row lq, pieces 2 s + lh.  V (transposed while it is read: sixteen lanes fetch 4 keys x 16
    // head dims and each ends up with the 4 keys of one dim): key 4 lh + (lane % 16) / 4, dims 16 ((lane / 16) % 2) + 4 (lane % 4) .. + 3.
    auto k_frag = [&](const uint8_t* tile, int h, int s) {
        return *reinterpret_cast<const v8h*>(tile + ((kh + h) * 32 + lq) * ROW + piece_of<HD>(lq, 2 * s + lh) * 16);
    };
    const uint32_t vrow = 4 * lh + ((lane & 15) >> 2), vpiece = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    auto v_at = [&](const uint8_t* tile, int key, int d) { return tile + vrow * ROW + piece_of<HD>(vrow, 4 * d + vpiece) * 16 + (lane & 1) * 8 + key * ROW; };
    auto v_frag = [&](const uint8_t* tile, int key, int d) {       // keys key + 4 lh .. + 3 and key + 8 + 4 lh .. + 3
        const uint8_t* at = v_at(tile, key, d);
        const v4h v0 = read_transposed(at), v1 = read_transposed(at + 8 * ROW);
        return (v8h){v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
    };

    load_tiles(tile0, tile0 & 1);
    if constexpr (!DIRECT) put_tiles(tile0 & 1);
    // ---- Q fragment (B operand of S^T = K Q^T): lane (lq, lh) holds q[row][16 s + 8 lh + 0..7].  All of it is requested at once (a row past the
    // last takes the last one's): with a condition around each load they waited for one another (3001 tokens of 32/32 heads of 96: 1.8 us more).
    v8h qf[NS];
    {
        const float4* p = reinterpret_cast<const float4*>(q + (size_t)min(qrow, M - 1) * q_stride + head * HD + 8 * lh);
        float4 f[NS][2];
#pragma unroll
        for (int s = 0; s < NS; s++) { f[s][0] = p[4 * s]; f[s][1] = p[4 * s + 1]; }
#pragma unroll
        for (int s = 0; s < NS; s++)
            qf[s] = (v8h){(_Float16)f[s][0].x, (_Float16)f[s][0].y, (_Float16)f[s][0].z, (_Float16)f[s][0].w,
                          (_Float16)f[s][1].x, (_Float16)f[s][1].y, (_Float16)f[s][1].z, (_Float16)f[s][1].w};
    }
    for (uint32_t kt = tile0; kt < ntiles; kt++) {
        const uint32_t buf = kt & 1;
        __builtin_amdgcn_s_waitcnt(0);       // this wave's share of the step's tiles is in LDS,
        __syncthreads();                     // and so is everyone's; nobody reads the other buffer any more
        if (kt + 1 < ntiles) load_tiles(kt + 1, buf ^ 1);
        const uint32_t k0 = kt * KT + kh * 32;            // this wave's first 32 keys of the tile
        constexpr uint32_t KW = 32 * KH;                  // keys of the tile this wave works
        if (wave_active && k0 <= wave_max_pos && k0 + KW > wave_lo) {   // else they lie entirely in the group's future, or before every window
            const uint8_t* Kb = smem + buf * 2 * TILE;
            const uint8_t* Vb = Kb + TILE;
            // ---- S^T tiles: sacc[h][r] = q . k for key k0 + 32 h + 8(r/4) + 4 lh + r%4, query lq
            v16f sacc[KH];
#pragma unroll
            for (int h = 0; h < KH; h++)
#pragma unroll
                for (int r = 0; r < 16; r++) sacc[h][r] = 0.f;
#pragma unroll
            for (int s = 0; s < NS; s++)
#pragma unroll
                for (int h = 0; h < KH; h++) {
                    sacc[h] = __builtin_amdgcn_mfma_f32_32x32x16_f16(k_frag(Kb, h, s), qf[s], sacc[h], 0, 0, 0);
                }
            // ---- causal mask: only keys past the group's first query can be masked for some query
            // with a window, also keys that the group's last query no longer sees
#pragma unroll
            for (int h = 0; h < KH; h++) {
                const uint32_t kb = k0 + 32 * h;
                if (WIN && (kb + 31 > wave_min_pos || kb + window <= wave_max_pos)) {
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const uint32_t t = kb + 8 * (r >> 2) + 4 * lh + (r & 3);
                        sacc[h][r] = (t <= qpos && t + window > qpos) ? sacc[h][r] : -INFINITY;
                    }
                } else if (!WIN && kb + 31 > wave_min_pos) {
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const uint32_t t = kb + 8 * (r >> 2) + 4 * lh + (r & 3);
                        sacc[h][r] = (t <= qpos) ? sacc[h][r] : -INFINITY;
                    }
                }
            }
            // ---- online softmax in base 2 (per-lane scalars: a lane owns one query)
            float m_tile = -INFINITY;
#pragma unroll
            for (int h = 0; h < KH; h++)
#pragma unroll
                for (int r = 0; r < 16; r++) m_tile = fmaxf(m_tile, sacc[h][r]);
            m_tile = lane_xor_max<32>(m_tile) * c2;      // c2 > 0: max commutes with the scaling
            const bool risen = m_tile > m_run;
            if (__builtin_amdgcn_ballot_w64(risen) != 0) {
                const float m_new = risen ? m_tile : m_run;
                const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
                l_run *= alpha;
#pragma unroll
                for (int d = 0; d < ND; d++)
#pragma unroll
                    for (int r = 0; r < 16; r++) oacc[d][r] *= alpha;
                m_run = m_new;
            }
            // a query that has seen no key yet (all of these keys masked for it) keeps m = -inf: exponentiate
            // against 0 instead, every p is then 2^-inf = 0
            const float m_exp = m_run == -INFINITY ? 0.f : m_run;
            float l_tile = 0.f;      // a tile's own: one by one onto the sum of thousands, weights that are alike are rounded alike
            v8h pb[KH][2];
#pragma unroll
            for (int h = 0; h < KH; h++)
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int e = 0; e < 8; e++) {
                        const float p = __builtin_amdgcn_exp2f(fmaf(sacc[h][8 * j + e], c2, -m_exp));   // 2^-inf = 0 for masked keys
                        l_tile += p;
                        pb[h][j][e] = (_Float16)p;
                    }
            l_run += l_tile;
            // ---- O^T += V^T P^T over this wave's keys
#pragma unroll
            for (int h = 0; h < KH; h++) {
                v8h vf[2][ND];
                if constexpr (OWN) read_v<HD>(vf, (uint32_t)(uintptr_t)FH_LDS3(v_at(Vb, (kh + h) * 32, 0)), (uint32_t)(uintptr_t)FH_LDS3(v_at(Vb, (kh + h) * 32, 1)));
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int d = 0; d < ND; d++) {
                        if constexpr (!OWN) vf[j][d] = v_frag(Vb, (kh + h) * 32 + 16 * j, d);
                        oacc[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[j][d], pb[h][j], oacc[d], 0, 0, 0);
                    }
            }
        }
        if constexpr (!DIRECT) {
            if (kt + 1 < ntiles) put_tiles(buf ^ 1);
        }
    }

    // ---- the two waves of a query group merge their halves: the odd one hands (m, l, O) over through LDS
    float* mg = reinterpret_cast<float*>(smem) + (qg * 64 + lane) * MERGE_FLOATS;
    if (KH == 1) {
    __syncthreads();          // the tile buffers are free
    if (kh == 1) {
        mg[0] = m_run;
        mg[1] = l_run;
#pragma unroll
        for (int d = 0; d < ND; d++)
#pragma unroll
            for (int r = 0; r < 16; r++) mg[2 + d * 16 + r] = oacc[d][r];
    }
    __syncthreads();
    if (kh == 1) return;
    {
        const float m1 = mg[0], l1 = mg[1];
        const float m = fmaxf(m_run, m1);            // finite: every query sees itself (without a window, key 0 in the even half too)
        const float a0 = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m), a1 = m1 == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m1 - m);
        l_run = l_run * a0 + l1 * a1;
#pragma unroll
        for (int d = 0; d < ND; d++)
#pragma unroll
            for (int r = 0; r < 16; r++) oacc[d][r] = oacc[d][r] * a0 + mg[2 + d * 16 + r] * a1;
    }
    }

    // ---- normalise and store: lane (lq, lh) holds out[qrow][32 d + 8 g + 4 lh + 0..3]
    const float l_tot = lane_xor_add<32>(l_run);
    if (QUANT) {
        const float inv_l = 1.0f / l_tot;
        const uint32_t width = heads * HD;
#pragma unroll
        for (int d = 0; d < ND; d++) {
            float o[16], amax = 0.f;
#pragma unroll
            for (int r = 0; r < 16; r++) { o[r] = oacc[d][r] * inv_l; amax = fmaxf(amax, fabsf(o[r])); }
            amax = lane_xor_max<32>(amax);
            float inv;
            const float sc = act_scale(amax, inv);
            // QUANT has no f32 output, so out_stride carries a flag instead: store the odd blocks of a row negated
            if (out_stride != 0 && ((head * (HD / 32) + d) & 1u) != 0) inv = -inv;
            if (qrow < M) {
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const uint32_t pk = ((uint32_t)quant_code(o[4 * g] * inv) & 0xFFu) | (((uint32_t)quant_code(o[4 * g + 1] * inv) & 0xFFu) << 8) |
                                        (((uint32_t)quant_code(o[4 * g + 2] * inv) & 0xFFu) << 16) | (((uint32_t)quant_code(o[4 * g + 3] * inv) & 0xFFu) << 24);
                    *reinterpret_cast<uint32_t*>(oq + (size_t)qrow * width + head * HD + 32 * d + 8 * g + 4 * lh) = pk;
                }
                // (for the fast GEMM an all-zero block carries the scale 0, see quantize_block_part)
                if (lh == 0) osc[(size_t)qrow * (width / 32) + head * (HD / 32) + d] = (out_stride != 0 && amax == 0.f) ? (uint16_t)0 : f32_to_f16_bits(sc);
            }
        }
        return;
    }
    if (qrow < M) {
        const float inv_l = 1.0f / l_tot;
        float* orow = out + (size_t)qrow * out_stride + head * HD;
#pragma unroll
        for (int d = 0; d < ND; d++)
#pragma unroll
            for (int g = 0; g < 4; g++) {
                float4 o = make_float4(oacc[d][4 * g] * inv_l, oacc[d][4 * g + 1] * inv_l, oacc[d][4 * g + 2] * inv_l,
                                       oacc[d][4 * g + 3] * inv_l);
                *reinterpret_cast<float4*>(orow + 32 * d + 8 * g + 4 * lh) = o;
            }
    }
}

namespace {
template <int HD, bool QUANT>
void launch_win(dim3 grid, hipStream_t s, const float* q, const uint16_t* kc, const uint16_t* vc, float* out, uint32_t q_stride,
                uint32_t out_stride, uint32_t M, uint32_t base_pos, uint32_t heads, uint32_t kv_heads, int8_t* oq, uint16_t* osc,
                uint32_t window, PageTable pt) {
    // The four-wave form where there are many workgroups: then throughput decides, and a wave with two score tiles per step does more of it; the eight-wave form below: then the
    // longest workgroup's chain of tile steps decides, and twice the waves halve its steps.  us, four waves / eight, heads of 64, 96, 128 (as they are taken: see own_waits):
    //   workgroups      384 (2000 rows of 24/8) 33.3 / 32.7, 40.9 / 40.0, 50.6 / 47.9    480 (2500) 41.0 / 41.2, 51.9 / 54.8, 64.2 / 65.7    768 (4000) 74.7 / 80.2, 97.7 / 121, 120 / 147
    //   under a window  180 (2500 rows of 9/3, 1500) 29.1 / 28.6, 35.5 / 34.2, 42.6 / 38.7    288 (1500 behind 1500 of 24/8, 700) 27.6 / 28.9, 35.3 / 44.4, 41.0 / 51.7
    //                   480 (2500 of 24/8, 256) 17.1 / 18.0, 22.5 / 29.5, 26.0 / 35.5    (2000) 38.3 / 39.2, 49.3 / 56.4, 60.1 / 66.0    320 (2500 of 16/16, 2000) 36.9 / 35.9,
    //                   45.6 / 42.6, 54.9 / 48.4
    // Short prompts would gain from four waves as well (300 rows of 24/8 7.8 / 9.4, 9.8 / 11.8, 11.4 / 14.0, 1000 18.4 / 19.5, 22.9 / 23.5, 27.5 / 27.5), unless they have few rows behind
    // many (33 behind 1400 of 9/3 23.0 / 18.8, 27.9 / 22.5, 33.8 / 23.4); but then the parts of one prompt would be worked on in different orders.  FORGE_HIP_ATTN_WAVES=8 / 4 forces one.
    static const int forced = [] { const char* e = getenv("FORGE_HIP_ATTN_WAVES"); return e ? atoi(e) : 0; }();
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n = 256;
        return n > 0 ? n : 256;
    }();
    // a window that covers every key of the call is plain causal attention
    const bool win = window != 0 && window < base_pos + M;
    const bool alike = win && window <= (base_pos + M) / 2;      // a narrow window makes nearly all workgroups equally long
    const bool many = alike ? grid.x > (uint32_t)cus : grid.x >= (uint32_t)cus * 7 / 4;
    const bool four = forced == 4 || (forced != 8 && many);
    // A model's caches are its own allocations; an operation's caller can have one that begins off a 16-byte boundary.  us, on one / 8 bytes off: 3001 rows of 32/32 heads of 96
    // 87.9 / 93.4, of 32/8 of 128 101 / 110, 2502 of 32/8 of 64 45.9 / 51.6.
    const bool direct = QUANT || ((reinterpret_cast<uintptr_t>(kc) | reinterpret_cast<uintptr_t>(vc)) & 15) == 0;
    auto go = [&](auto direct_) {
#define FH_AP(WIN_, KH_) \
    fh::launch(attn_prefill_kernel<HD, QUANT, WIN_, KH_, decltype(direct_)::value>, grid, AP_THREADS / KH_, 0, s, q, kc, vc, out, q_stride, out_stride, M, base_pos, heads, kv_heads, oq, osc, \
               WIN_ ? window : 0u, pt)
        if (win) { if (four) FH_AP(true, 2); else FH_AP(true, 1); }
        else { if (four) FH_AP(false, 2); else FH_AP(false, 1); }
#undef FH_AP
    };
    if (direct) go(std::true_type{});
    else if constexpr (!QUANT) go(std::false_type{});
}
template <bool QUANT>
void launch_hd(uint32_t hd, dim3 grid, hipStream_t s, const float* q, const uint16_t* kc, const uint16_t* vc, float* out,
               uint32_t q_stride, uint32_t out_stride, uint32_t M, uint32_t base_pos, uint32_t heads, uint32_t kv_heads, int8_t* oq,
               uint16_t* osc, uint32_t window, PageTable pt) {
    if (hd == 64) launch_win<64, QUANT>(grid, s, q, kc, vc, out, q_stride, out_stride, M, base_pos, heads, kv_heads, oq, osc, window, pt);
    else if (hd == 96) launch_win<96, QUANT>(grid, s, q, kc, vc, out, q_stride, out_stride, M, base_pos, heads, kv_heads, oq, osc, window, pt);
    else launch_win<128, QUANT>(grid, s, q, kc, vc, out, q_stride, out_stride, M, base_pos, heads, kv_heads, oq, osc, window, pt);
}
}  // namespace

void launch_attn_prefill(const float* q, uint32_t q_stride, const uint16_t* kc, const uint16_t* vc, float* out,
                         uint32_t out_stride, uint32_t M, uint32_t base_pos, uint32_t heads, uint32_t kv_heads,
                         uint32_t hd, uint32_t window, hipStream_t s, PageTable pt) {
    if (M == 0) return;
    dim3 grid(((M + QB - 1) / QB) * heads);
    launch_hd<false>(hd, grid, s, q, kc, vc, out, q_stride, out_stride, M, base_pos, heads, kv_heads, nullptr, nullptr, window, pt);
}

void launch_attn_prefill_quant(const float* q, uint32_t q_stride, const uint16_t* kc, const uint16_t* vc, int8_t* oq, uint16_t* osc,
                               uint32_t M, uint32_t base_pos, uint32_t heads, uint32_t kv_heads, uint32_t hd, uint32_t window,
                               hipStream_t s, bool neg_odd, PageTable pt) {
    if (M == 0) return;
    dim3 grid(((M + QB - 1) / QB) * heads);
    launch_hd<true>(hd, grid, s, q, kc, vc, nullptr, q_stride, neg_odd ? 1u : 0u, M, base_pos, heads, kv_heads, oq, osc, window, pt);
}

}  // namespace fh
