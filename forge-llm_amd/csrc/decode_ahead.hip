// One decode token as ONE kernel whose waves hold their share of a layer's matrices in registers (model::forward, emit.rs:4029-4227).
//
// A step is a chain of four products and an attention per layer.  As kernels a link of that chain is 4 to 6 us however small (a launch that does nothing takes
// 2.7); as phases of the kernel that streams weights of any size (decode_persistent.hip) it is 5.  Here a layer of SmolLM2-135M takes 12 us, one of the 1B shape 21
// (its 65 MB alone take 13): five hand-overs of 0.8 to 1.2 (1.5 to 2.5 beside weights), two norms of 0.7, attention 3.2, and the products.
//   * A wave's rows are a few registers, requested where nothing is on its way to the compute unit: while the attention is at work, and with wide models also right
//     behind the products.  (A compute unit's loads return in order and its queue is short: a poll behind weights comes when they have come, and so does a store.)
//   * Eight waves hold weights, four fetch the vectors.  A wave forms and sums whole rows by itself; the workgroup's rows lie side by side and are handed over
//     by ONE store.  (Element by element from eight waves a hand-over of 576 elements among 72 workgroups takes 1.9 us, by one store 1.2; among 144 workgroups 1.5, among 256
//     1.8: hence no more workgroups than the rows need.)
//   * A polling thread requests all its elements before it looks at one, without a condition around a load (behind which the compiler would wait for it).
//   * Attention workgroups request a head's cached rows a layer ahead.
//   * Pointers come from a copy in LDS: a scalar load of a line that nobody has touched takes a microsecond.
// Values travel between workgroups as tagged 8-byte elements (resident.h; every wait is bounded, as in decode_persistent.hip): a buffer is overwritten only by a
// phase whose inputs transitively depend on every reader of what it held.
//
// ORD: the arithmetic in the reference's own order (block products, row sums, norm, softmax over 64-key blocks, the C library's expf), bit-identical to the
// order-faithful kernel sequence; narrow models, to which the order costs nothing, run it in both modes.  Otherwise row sums and the norm's sum add up as the lanes
// have them.  Per token in us, kernel sequence (order-faithful mode) / decode_persistent.hip (fast mode) / this, by rows of context:
//   SmolLM2-135M Q8_0   33: 781 / 880 / 384    300: 820 / 878 / 421    740: 907 / 876 / 466
//   1B shape Q8_0       33: 754 / 610 / 450 and 400 (order-faithful, fast)    200: - / 636 / 458 and 420       Q4_0, fast: 33: 532 / 403
//   and in fast mode (PaPart) 300: 637 / 442    1000: 642 / 447    2400: 644 / 459    5000: 676 / 495    Q4_0 2400: 570 / 441
//   and of Q4_K / Q6_K matrices (llama.cpp's Q4_K_M recipe), 1B shape 33: 623 / 457    300: 646 / 495    2400: 655 / 511    5000: 688 / 548
// Heads of 96 and 128 gain as much though those of 128 spill (8 layers, 33 rows, fast: 8/2 of 96 at 768 channels 213 / 136, 6/2 of 128 207 / 138, 16/4 of 96 at 1536 246 / 174,
// 12/4 of 128 at 1024 212 / 168).  The chain takes the time, as far as a layer's weights arrive
// beside it: half the bytes make no layer shorter (1B shape, us: Q8_0 21, Q4_0 21), an earlier request for those that were waited for did (Q8_0 23 -> 21: EARLY).
#include <stddef.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <memory>
#include <vector>

#include "attn_decode_math.h"
#include "common.h"
#include "device_utils.h"
#include "expf_ref.h"
#include "gemv_order.h"
#include "resident.h"
#include "resident_seat.h"

namespace fh {

namespace {

constexpr uint32_t PA_POLL = 4, PA_COMP = 8, PA_WAVES = PA_POLL + PA_COMP, PA_THREADS = PA_WAVES * 64, PA_POLL_THREADS = PA_POLL * 64;
constexpr uint32_t PA_B = 64;                 // FLASH_ATTN_BLOCK_SIZE, emit.rs:201; a wave takes one block of keys: at most PA_WAVES blocks
constexpr uint32_t PA_MAX_ROWS = 8;           // rows of a product that one wave holds (not the lm_head)
constexpr uint32_t PA_SUM = 24, PA_SSQ = 12;  // a row's products, and an accumulator's elements of the norm, are read in groups of so many: LDS rows end in zeros up to there
// The two forms.  UQ .. UL: blocks of 32 weights that a lane holds of q;k;v, o, gate;up (two sets), down and each of two sets of the lm_head; NX, NV: elements
// a polling thread takes of the residual row and of gate;up's quantised vector; AW: waves that attend to a head, each to 64 keys.
//   Narrow (up to 768 channels): a layer in 54 registers of a few dozen workgroups; the heads have workgroups of their own, up to 768 rows of context.
//   Wide (up to 2048 channels): every compute unit holds a block of 32 gate;up rows in two sets of registers, so heads and weights share workgroups: the last `heads` of
//   them hold no rows of q;k;v and o, and their fetching waves attend, to up to 256 rows (longer contexts, order free: every workgroup's, PaPart).  down takes the place of one of them when that is done.
struct PaNarrow { static constexpr int UQ = 1, UO = 1, UG1 = 3, UG2 = 0, UD = 1, UL = 4, NX = 3, NV = 3; static constexpr uint32_t AW = PA_WAVES; static constexpr bool WIDE = false; };
struct PaWide { static constexpr int UQ = 2, UO = 2, UG1 = 4, UG2 = 4, UD = 4, UL = 4, NX = 8, NV = 9; static constexpr uint32_t AW = PA_POLL; static constexpr bool WIDE = true; };

// How a matrix's blocks of 32 weights lie in memory.  Q8, Q4: as for every other kernel.  KQ: Q4_K and Q6_K alike, made by pa_create: the codes as int8 in order
// (0 .. 15 and -32 .. 31) and a word: fp16 bits of d (Q4_K, odd blocks: of dmin) | an int8 scale << 16 | Q6_K: the second half's << 24, Q4_K: the minimum << 24.
// (One form for both, twice the bytes that Q4_K's codes need.  4 bits in a form of their own were not measured.)
enum PaFmt : int { PA_Q8, PA_Q4, PA_KQ };

// magic: floor(2^32 / nblk) + 1; R: rows per wave; wg0: the first workgroup with rows; stride: words between two rows of products; prod: the first wave's area of
// them (LDS bytes), dump: a word behind it that nobody reads; fold: log2 of the lanes that add a row up where the order is free
struct PaMat { uint32_t N, nblk, magic, R, wg0, stride, prod, dump, fold; };
struct PaWeights { const uint8_t* qs; const uint16_t* ws; };
struct PaLayer {
    PaWeights w[4];                           // q;k;v, o, gate;up, down
    const float* norm[2];
    uint16_t* kc;
    uint16_t* vc;
};

struct PaArgs {
    PaMat m[5];                               // q;k;v, o, gate;up (N = 2 I; a workgroup holds 32 + 32 rows), down, lm_head
    uint32_t L, H, I, QKS, KV, heads, kv_heads;
    const uint32_t* pages;                    // paged cache: pool page of each page of the sequence (null: rows lie in order); a page has at least PA_B rows
    uint32_t page_shift, n_pages;
    uint32_t splits;                          // Wide, order free: parts that a long context is attended in (0: it is not)
    uint32_t G, head0;                        // workgroups [0, G) hold the layers' matrices, [head0, head0 + heads) take a head each; all share the lm_head
    float eps;
    const PaLayer* layers;                    // [L + 1]: the last one's first norm is the final norm; its q;k;v is the first layer's (requested, not used)
    PaWeights lm;
    const float* embed;
    const float* cos_t;
    const float* sin_t;
    // tagged exchange buffers
    uint64_t* tx;      // [H]                residual stream
    uint64_t* tq;      // [QKS]              rotated q
    uint64_t* tkv;     // [2 KV]             this position's K row (rotated) and V row, fp16 bits
    uint64_t* taq;     // [QKS/32][9]        attention output, a block of 32: int8 codes (4 per element), then the fp16 scale
    uint64_t* taq2;    // [I/32][9]          silu(gate)*up, same format
    uint64_t* trec;    // [heads][splits][HD + 2]  Wide, long contexts: a split's weighted sum, maximum and weight sum
    uint64_t* tpart;   // [2 workgroups of the grid]  argmax candidates
    float* logits;
    uint32_t* state;   // [0] position  [1] token  [2] next token  [3] abort flag  [4] number of the step that counted its token
    uint32_t* counts;
    float penalty;
    uint32_t tag_base, spin_limit, token, step_seq;
    unsigned long long* host_out;             // host-mapped {launch number, next token}: written last, or null
    uint32_t host_seq;
    unsigned long long* stamps;               // optional: wall clock between the phases, each from a workgroup that has done the phase before
    uint32_t off_as, off_xs, off_out, off_silu, off_prod, off_layers, off_attn, off_rec, prod_words, lds_words, xstride;      // LDS byte offsets (activation codes at 0)
    uint32_t to_sums;                         // KQ: from the activation scales to the blocks' sums of codes
    uint32_t six[5], six_v;                   // KQ: which matrices are Q6_K; the v rows of q;k;v have a format of their own
};

// A uniform base and a lane's 32-bit offset in bytes.
template <typename T>
__device__ __forceinline__ T pa_at(const void* base, uint32_t off) { return ldg(reinterpret_cast<const T*>(static_cast<const uint8_t*>(base) + off)); }

// Pointers of a layer, from their copy in LDS (a scalar load of a line that nobody has touched takes a microsecond).
template <typename T>
__device__ __forceinline__ T pa_lds_ptr(const T& p) {
    const uint64_t v = *reinterpret_cast<const uint64_t*>(&p);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)v), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(v >> 32));
    return reinterpret_cast<T>(((uint64_t)hi << 32) | lo);
}
__device__ __forceinline__ PaWeights pa_lds_ptr(const PaWeights& w) { return PaWeights{pa_lds_ptr(w.qs), pa_lds_ptr(w.ws)}; }

__host__ __device__ constexpr uint32_t pa_up(uint32_t v, uint32_t m) { return (v + m - 1) / m * m; }

// A wave's blocks of a matrix: n of them, row after row; from block `seg` on they lie `jump` blocks further (the up rows of gate;up).
// six: KQ, 1 for Q6_K.
struct PaTask { uint32_t base, n, seg, jump, six; };
__device__ __forceinline__ uint32_t pa_sgpr(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
__device__ __forceinline__ uint32_t pa_rows(const PaMat& m, uint32_t wv) { return wv * m.R < m.N ? min(m.R, m.N - wv * m.R) : 0u; }
__device__ __forceinline__ PaTask pa_task(const PaMat& m, uint32_t wv, uint32_t six = 0) {
    const uint32_t rows = pa_rows(m, wv);
    return PaTask{rows ? wv * m.R * m.nblk : 0u, rows * m.nblk, 0xFFFFFFFFu, 0u, six};
}

// Lane l of round j holds block 64 j + l (Q4), or halves of two blocks (Q8, KQ): of blocks 64 j + l / 2 and 64 j + 32 + l / 2 the half
// l & 1, so that a load covers consecutive bytes; the sums of both halves meet by a move between neighbours.
template <int U, PaFmt W> struct PaSet { int4 v[W == PA_Q4 ? U : 2 * U]; uint32_t s[U]; };
template <PaFmt W>
__device__ __forceinline__ uint32_t pa_own(uint32_t j, uint32_t lane) { return W == PA_Q4 ? 64 * j + lane : 64 * j + 32 * (lane & 1u) + (lane >> 1); }

// [A, B): the rounds of the set that are requested (B = -1: up to its last).
template <int J0 = 0, int A = 0, int B = -1, int U, PaFmt W>
__device__ __forceinline__ void pa_load(PaSet<U, W>& w, const PaWeights& mat, const PaTask& t, uint32_t lane) {
    asm volatile("" : "+v"(lane));           // the addresses are worked out here: kept from layer to layer they would not fit the registers
    // Blocks past the last one re-read it, and a wave without rows reads the matrix's first block: with no condition around them the loads in flight are
    // known where a product waits for its own.
    const uint32_t last = max(t.n, 1u) - 1;
    auto at = [&](uint32_t unit) {
        const uint32_t u = min(unit, last);
        return t.base + u + (u >= t.seg ? t.jump : 0u);
    };
#pragma unroll
    for (int j = A; j < (B < 0 ? U : B); j++) {
        if (W == PA_Q4) {
            w.v[j] = pa_at<int4>(mat.qs, at(64 * (J0 + j) + lane) * 16);
        } else {
#pragma unroll
            for (int h = 0; h < 2; h++) w.v[2 * j + h] = pa_at<int4>(mat.qs, at(64 * (J0 + j) + 32 * h + (lane >> 1)) * 32 + (lane & 1u) * 16);
        }
        if constexpr (W == PA_KQ) w.s[j] = pa_at<uint32_t>(mat.ws, at(pa_own<W>(J0 + j, lane)) * 4);
        else w.s[j] = pa_at<uint16_t>(mat.ws, at(pa_own<W>(J0 + j, lane)) * 2);
    }
}

// Where a lane finds its blocks' activations and leaves their products (LDS bytes), worked out ahead of the wait for the vector.
template <int U, PaFmt W> struct PaIdx { uint32_t a[W == PA_Q4 ? U : 2 * U], s[U], p[U]; };
template <int U, PaFmt W, int J0 = 0>
__device__ __forceinline__ PaIdx<U, W> pa_index(const PaTask& t, const PaMat& m, uint32_t off_as, uint32_t prod, uint32_t lane) {
    PaIdx<U, W> x;
#pragma unroll
    for (int j = 0; j < U; j++) {
        const uint32_t u = pa_own<W>(J0 + j, lane), r = __umulhi(u, m.magic), b = u - r * m.nblk;      // b is a block of the row whatever u is
        x.s[j] = off_as + b * 4;
        x.p[j] = u < t.n ? prod + (r * m.stride + b) * 4 : prod + m.dump;
        if (W == PA_Q4) {
            x.a[j] = b * 32;
        } else {
#pragma unroll
            for (int h = 0; h < 2; h++) {
                const uint32_t uh = 64 * (J0 + j) + 32 * h + (lane >> 1);
                x.a[2 * j + h] = (uh - __umulhi(uh, m.magic) * m.nblk) * 32 + (lane & 1u) * 16;
            }
        }
        asm volatile("" : "+v"(x.s[j]), "+v"(x.p[j]));
    }
#pragma unroll
    for (int i = 0; i < (W == PA_Q4 ? U : 2 * U); i++) asm volatile("" : "+v"(x.a[i]));
    return x;
}

// The blocks' products, parked in the wave's LDS: (a_s * w_s) * f32(isum) of an exact int32 block sum, or the block's term of dot_q4_k_q8_0 / dot_q6_k_q8_0
// (emit.rs:3035-3306, 3553-3612), a_s * (d * f32(sum of scale * isum over the halves) - (dmin * minimum) * f32(sum of the codes)): both sums whole numbers of less than
// 2^24.  sums: KQ, from a block's activation scale to the sum of its codes (LDS bytes).
template <int J0 = 0, int U, PaFmt W>
__device__ __forceinline__ void pa_products(const PaSet<U, W>& w, const PaIdx<U, W>& x, const PaTask& t, uint8_t* smem, uint32_t sums) {
#pragma unroll
    for (int j = 0; j < U; j++) {
        if (64u * (J0 + j) >= t.n) break;
        int isum;
        if (W == PA_Q4) {
            const int4 a0 = *reinterpret_cast<const int4*>(smem + x.a[j]);
            const int4 a1 = *reinterpret_cast<const int4*>(smem + x.a[j] + 16);
            const int4 v = w.v[j];
            const int k = 0x0F0F0F0F;
            const int4 lo = make_int4(v.x & k, v.y & k, v.z & k, v.w & k);
            const int4 hi = make_int4((v.x >> 4) & k, (v.y >> 4) & k, (v.z >> 4) & k, (v.w >> 4) & k);
            const int4 ones = make_int4(0x01010101, 0x01010101, 0x01010101, 0x01010101);
            isum = dot16(hi, a1, dot16(lo, a0, 0)) - 8 * dot16(ones, a1, dot16(ones, a0, 0));
        } else {
            int d[2];
#pragma unroll
            for (int h = 0; h < 2; h++) d[h] = dot16(w.v[2 * j + h], *reinterpret_cast<const int4*>(smem + x.a[2 * j + h]), 0);
            if constexpr (W == PA_KQ) {
                // this lane's half of either block times its scale: its own block's word and its neighbour's
                const bool odd = __lane_id() & 1u;
                const uint32_t own = w.s[j], far = lane_xor<1>(own), up = odd && t.six ? 0u : 8u;
                d[0] = __mul24(d[0], (int)((odd ? far : own) << up) >> 24);
                d[1] = __mul24(d[1], (int)((odd ? own : far) << up) >> 24);
            }
#pragma unroll
            for (int h = 0; h < 2; h++) d[h] += lane_xor<1>(d[h]);
            isum = (__lane_id() & 1u) ? d[1] : d[0];
        }
        const float as = *reinterpret_cast<const float*>(smem + x.s[j]);
        float* p = reinterpret_cast<float*>(smem + x.p[j]);
        if constexpr (W == PA_KQ) {
            // d and dmin of a super-block lie in its even and odd blocks
            const uint32_t own = w.s[j], mate = lane_xor<2>(own);
            const bool second = __lane_id() & 2u;
            const float d = f16_bits_to_f32((uint16_t)(second ? mate : own)), dmin = f16_bits_to_f32((uint16_t)(second ? own : mate));
            const float asum = *reinterpret_cast<const float*>(smem + x.s[j] + sums);
            *p = as * (d * (float)isum - (t.six ? 0.f : dmin * (float)(own >> 24)) * asum);
        } else {
            *p = (as * f16_bits_to_f32((uint16_t)w.s[j])) * (float)isum;
        }
    }
}

// Sums of the wave's rows.  Products and sums are one wave's LDS operations, which execute in order.
//   ORD      in block order: lane r < rows holds row r's.  The zeros behind a row's products change nothing: a sum that starts at +0 is never -0.
//   not ORD  2^fold lanes add a row up (as many as there are for m.R rows), the first of them holds it.
struct PaSum { float v; uint32_t row; bool on; };
template <bool ORD>
__device__ __forceinline__ PaSum pa_row_sum(const PaMat& m, uint32_t rows, const uint8_t* area, uint32_t lane) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if constexpr (!ORD) {
        const uint32_t row = lane >> m.fold, part = lane & ((1u << m.fold) - 1);
        const float* p = reinterpret_cast<const float*>(area) + row * m.stride;
        float r = 0.f;
        for (uint32_t b = part; b < m.nblk; b += 1u << m.fold) r += p[b];
        if (m.fold > 0) r = lane_xor_add<1>(r);
        if (m.fold > 1) r = lane_xor_add<2>(r);
        if (m.fold > 2) r = lane_xor_add<4>(r);
        if (m.fold > 3) r = lane_xor_add<8>(r);
        if (m.fold > 4) r = lane_xor_add<16>(r);
        if (m.fold > 5) r = lane_xor_add<32>(r);
        return PaSum{r, row, part == 0 && row < rows};
    }
    float r = 0.f;
    if (lane < rows) {
        const float4* p = reinterpret_cast<const float4*>(area) + lane * (m.stride / 4);
        constexpr int N4 = PA_SUM / 4;
        float4 v[N4], w[N4];
#pragma unroll
        for (int i = 0; i < N4; i++) v[i] = p[i];
        for (uint32_t b = PA_SUM; b < m.nblk; b += PA_SUM) {
            p += N4;
#pragma unroll
            for (int i = 0; i < N4; i++) w[i] = p[i];
#pragma unroll
            for (int i = 0; i < N4; i++) { r = r + v[i].x; r = r + v[i].y; r = r + v[i].z; r = r + v[i].w; }
#pragma unroll
            for (int i = 0; i < N4; i++) v[i] = w[i];
        }
#pragma unroll
        for (int i = 0; i < N4; i++) { r = r + v[i].x; r = r + v[i].y; r = r + v[i].z; r = r + v[i].w; }
    }
    return PaSum{r, lane, lane < rows};
}

// int8 codes of 32 values, one per lane of a half wave, and their fp16 scale (emit.rs:1410-1440), as the nine elements of a block: side by side and by one
// instruction.  (Elements of one line that arrive one by one, from eight waves or with the scales elsewhere, cost the hand-over 0.7 us.)
// SUMS: the sum of the codes above the scale.
template <bool SUMS>
__device__ __forceinline__ void pa_store_block(float o, uint64_t* block, uint32_t tag, uint32_t lane, bool on) {
    const float amax = half_wave_max(fabsf(o));
    float inv;
    const float sc = act_scale(amax, inv);
    const uint32_t code = (uint32_t)quant_code(o * inv) & 0xFFu;
    const uint32_t pk = quad_broadcast<0>(code) | (quad_broadcast<1>(code) << 8) | (quad_broadcast<2>(code) << 16) | (quad_broadcast<3>(code) << 24);
    const uint32_t l = lane & 31u;            // lanes 0, 4, .. 28: codes; lane 1: the scale
    uint32_t last = f32_to_f16_bits(sc);
    if constexpr (SUMS) {
        int sum = __builtin_amdgcn_sdot4((int)pk, 0x01010101, 0, false);
        sum += lane_xor<4>(sum); sum += lane_xor<8>(sum); sum += lane_xor<16>(sum);
        last |= (uint32_t)sum << 16;
    }
    if (on && ((l & 3u) == 0 || l == 1)) stc64(block + (l == 1 ? 8u : l / 4), tag, l == 1 ? last : pk);
}

// Vectors, fetched by the polling waves.  The residual row lies in LDS accumulator by accumulator of the norm: element e in row e % 16.
__device__ __forceinline__ uint32_t pa_xs(uint32_t e, uint32_t xstride) { return (e & 15u) * xstride + (e >> 4); }
// Where the order of the norm's sum is free, every wave leaves the sum of its elements' squares in `part`.
template <int N, bool ORD>
__device__ __forceinline__ void pa_fetch_x(const uint64_t* tx, uint32_t tag, const float* emb, uint32_t H, float* xs, uint32_t xstride, float* part, const PollCtx& cx) {
    uint32_t v[N];
    if (!tag) {                               // the layer ahead of the first: the embedding row
#pragma unroll
        for (int i = 0; i < N; i++) v[i] = __float_as_uint(ldg(emb + min(cx.tid + i * PA_POLL_THREADS, H - 1)));
    } else {
        poll_tagged<N>([&](int i) { return tx + min(cx.tid + i * PA_POLL_THREADS, H - 1); }, [&](int) { return tag; }, v, cx);
    }
    float ss = 0.f;
#pragma unroll
    for (int i = 0; i < N; i++) {
        const uint32_t e = cx.tid + i * PA_POLL_THREADS;
        const float x = __uint_as_float(v[i]);
        if (e < H) {
            xs[pa_xs(e, xstride)] = x;
            ss = fmaf(x, x, ss);
        }
    }
    if constexpr (!ORD) {
        ss = wave_sum(ss);
        if (cx.lane == 0) part[cx.wave] = ss;
    }
}

// A quantised vector and, with it, the residual of the rows that this workgroup holds: element res_row of x in lane r of the first wave
// (res_tag 0: the embedding row; threads without a row: anything).
template <int NV, bool SUMS>
__device__ __forceinline__ float pa_fetch_aq(const uint64_t* t, uint32_t tag, uint32_t K, uint32_t* aq, float* as, float* sums, bool has_res, uint32_t res_row, const uint64_t* tx,
                                             uint32_t res_tag, const float* emb, const PollCtx& cx) {
    const uint32_t ne = K / 32 * 9;
    float re = 0.f;
    if (has_res && !res_tag) re = ldg(emb + res_row);
    // the residual is the last slot, with a tag of its own (it was final before the vector's phase began)
    const bool poll_res = has_res && res_tag != 0;
    const uint64_t* pr = poll_res ? tx + res_row : t;
    const uint32_t tr = poll_res ? res_tag : tag;
    auto fetch = [&](auto n) {
        constexpr int N = decltype(n)::value;
        uint32_t v[N + 1];
        poll_tagged<N + 1>([&](int i) { return i < N ? t + min(cx.tid + i * PA_POLL_THREADS, ne - 1) : pr; }, [&](int i) { return i < N ? tag : tr; }, v, cx);
#pragma unroll
        for (int i = 0; i < N; i++) {
            const uint32_t e = cx.tid + i * PA_POLL_THREADS, b = e / 9, k = e - b * 9;
            if (e < ne) {
                if (k < 8) aq[b * 8 + k] = v[i];
                else as[b] = f16_bits_to_f32((uint16_t)v[i]);
                if (SUMS && k == 8) sums[b] = (float)((int)v[i] >> 16);
            }
        }
        if (poll_res) re = __uint_as_float(v[N]);
    };
    if (ne <= PA_POLL_THREADS) fetch(std::integral_constant<int, 1>{});
    else if (ne <= 2 * PA_POLL_THREADS) fetch(std::integral_constant<int, 2>{});
    else if (NV == 3 || ne <= 3 * PA_POLL_THREADS) fetch(std::integral_constant<int, 3>{});
    else fetch(std::integral_constant<int, NV>{});
    return re;
}

// rms_norm (emit.rs:327-334) + activation quantiser.  In the reference's order (16 accumulators, emit.rs:272-295) each fetching wave walks the row and the first
// leaves 1 / rms behind; zeros behind an accumulator's elements change nothing.  The computing waves, which have nothing else to do yet, quantise four elements a
// thread, whose norm weights they hold.  (All twelve waves forming the sum for themselves and an element a thread: 1.1 us at 576 channels where this takes 0.7.)
__device__ __forceinline__ void pa_norm_sum(const float* xs, uint32_t xstride, float eps, uint32_t H, float* part, const PollCtx& cx) {
    const float4* p = reinterpret_cast<const float4*>(xs + (cx.lane & 15u) * xstride);
    float s = 0.f;
    constexpr int N4 = PA_SSQ / 4;
    float4 v[N4], w[N4];
#pragma unroll
    for (int i = 0; i < N4; i++) v[i] = p[i];
    for (uint32_t c = PA_SSQ; c < H / 16; c += PA_SSQ) {
        p += N4;
#pragma unroll
        for (int i = 0; i < N4; i++) w[i] = p[i];
#pragma unroll
        for (int i = 0; i < N4; i++) { s = fmaf(v[i].x, v[i].x, s); s = fmaf(v[i].y, v[i].y, s); s = fmaf(v[i].z, v[i].z, s); s = fmaf(v[i].w, v[i].w, s); }
#pragma unroll
        for (int i = 0; i < N4; i++) v[i] = w[i];
    }
#pragma unroll
    for (int i = 0; i < N4; i++) { s = fmaf(v[i].x, v[i].x, s); s = fmaf(v[i].y, v[i].y, s); s = fmaf(v[i].z, v[i].z, s); s = fmaf(v[i].w, v[i].w, s); }
    // (p[i] + p[4+i]) + (p[8+i] + p[12+i]) for i = 0..3, then (t0 + t1) + (t2 + t3): a pair's sum is the same in both of its lanes
    s = lane_xor_add<4>(s);
    s = lane_xor_add<8>(s);
    s = lane_xor_add<1>(s);
    s = lane_xor_add<2>(s);
    if (cx.tid == 0) part[0] = 1.0f / sqrtf(s / (float)H + eps);
}
template <bool ORD, bool SUMS>
__device__ __forceinline__ void pa_norm_quant(const float* xs, uint32_t xstride, float4 nw, float eps, uint32_t H, uint8_t* smem, uint32_t off_as, uint32_t to_sums, const float* part,
                                              uint32_t t) {
    if (t * 4 >= H) return;
    const float* p = xs + (t * 4 & 15u) * xstride + t / 4;        // four neighbours: rows t * 4 % 16 .. + 3
    const float x0 = p[0], x1 = p[xstride], x2 = p[2 * xstride], x3 = p[3 * xstride];
    const float inv_rms = ORD ? part[0] : 1.0f / sqrtf(((part[0] + part[1]) + (part[2] + part[3])) / (float)H + eps);
    const float4 v = make_float4(x0 * inv_rms * nw.x, x1 * inv_rms * nw.y, x2 * inv_rms * nw.z, x3 * inv_rms * nw.w);
    uint16_t sb;
    const uint32_t codes = quantize_block_part(v, sb);
    reinterpret_cast<uint32_t*>(smem)[t] = codes;
    if ((t & 7u) == 0) *reinterpret_cast<float*>(smem + off_as + t / 2) = f16_bits_to_f32(sb);
    if constexpr (SUMS) {
        int sum = __builtin_amdgcn_sdot4((int)codes, 0x01010101, 0, false);
        sum += lane_xor<1>(sum); sum += lane_xor<2>(sum); sum += lane_xor<4>(sum);
        if ((t & 7u) == 0) *reinterpret_cast<float*>(smem + off_as + t / 2 + to_sums) = (float)sum;
    }
}

struct PaExpTab {
    const uint64_t* p;
    __device__ __forceinline__ uint64_t operator()(int i) const { return p[i]; }
};

// LDS of an attention workgroup.  pn: products of q and this position's K row, vn: its V row, es: exp(m of the block before - m).
template <int HD, uint32_t AW>
struct PaAttn {
    float q[HD], pn[HD], vn[HD];
    float e[AW][PA_B];
    float sums[AW][HD];
    float bmax[AW], lblk[AW], es[AW], snew;
};

// A wave's 64-key block of the cache: lane = key of the K rows, lane = head dim of the V rows.  Heads of 64: all of it, in 32-bit; wider heads:
// K rows as they are and KC of the V rows at a time.
template <int HD>
struct PaKv {
    static constexpr int DPL = (HD + 63) / 64, KC = HD == 64 ? 64 : 16;
    float k[HD == 64 ? 64 : 1];
    uint4 kr[HD == 64 ? 1 : HD / 8];
    uint32_t v[KC / 2][DPL];                  // two rows to a register
    __device__ __forceinline__ void set_keys(const uint4 (&raw)[HD / 8]) {
#pragma unroll
        for (int c = 0; c < HD / 8; c++) {
            if constexpr (HD == 64) {
                const uint32_t w[4] = {raw[c].x, raw[c].y, raw[c].z, raw[c].w};
#pragma unroll
                for (int j = 0; j < 8; j++) k[c * 8 + j] = f16_bits_to_f32((uint16_t)(j & 1 ? w[j / 2] >> 16 : w[j / 2] & 0xFFFFu));
            } else {
                kr[c] = raw[c];
            }
        }
    }
    __device__ __forceinline__ float value(int i, int t) const { return f16_bits_to_f32((uint16_t)(i & 1 ? v[i / 2][t] >> 16 : v[i / 2][t] & 0xFFFFu)); }
    __device__ __forceinline__ float key(int i) const {
        if constexpr (HD == 64) {
            return k[i];
        } else {
            const uint4 r = kr[i / 8];
            const uint32_t w = i % 8 / 2 == 0 ? r.x : i % 8 / 2 == 1 ? r.y : i % 8 / 2 == 2 ? r.z : r.w;
            return f16_bits_to_f32((uint16_t)(i & 1 ? w >> 16 : w & 0xFFFFu));
        }
    }
};
// Where row t of the cache lies.
__device__ __forceinline__ uint32_t pa_row(const PaArgs& a, uint32_t t) {
    return a.pages ? (a.pages[t >> a.page_shift] << a.page_shift) + (t & ((1u << a.page_shift) - 1u)) : t;
}
// KC rows of V from row bs + k0 on, as they arrive: 16 bits to a register.  (Loads into halves of registers wait for each other in pairs.)
template <int HD> struct PaRaw { uint32_t v[PaKv<HD>::KC][PaKv<HD>::DPL]; };
template <int HD>
__device__ __forceinline__ void pa_load_values(PaRaw<HD>& raw, const uint16_t* vb, uint32_t row0, uint32_t pos, uint32_t delta, uint32_t zero, uint32_t kv_stride, uint32_t lane) {
#pragma unroll
    for (int i = 0; i < PaKv<HD>::KC; i++)
#pragma unroll
        for (int t = 0; t < PaKv<HD>::DPL; t++) {
            const uint32_t d = min(lane + 64 * t, (uint32_t)HD - 1), row = row0 + i;      // rows past the last cached one: the first
            raw.v[i][t] = pa_at<uint16_t>(vb + (row < pos ? row + delta : zero) * kv_stride, d * 2);
        }
    __builtin_amdgcn_sched_barrier(0);                // all requested before the first is waited for
}
template <int HD>
__device__ __forceinline__ void pa_pack_values(PaKv<HD>& kv, const PaRaw<HD>& raw) {
#pragma unroll
    for (int i = 0; i < PaKv<HD>::KC; i += 2)
#pragma unroll
        for (int t = 0; t < PaKv<HD>::DPL; t++) kv.v[i / 2][t] = raw.v[i][t] | (raw.v[i + 1][t] << 16);
    __builtin_amdgcn_sched_barrier(0);
}

// attention_flash (emit.rs:656-715) of one head, a wave per block of 64 keys: attn_exact_decode_one_kernel's steps.  AW waves attend, the workgroup's others only take
// part in the barriers.
template <int HD, uint32_t AW>
struct PaHead {
    uint32_t h, kvh, b, nb, bs, bl, nk;           // the wave's block b: bl keys, nk of them cached
    uint32_t delta, zero;                         // from a row of the block to where it lies; where the first row lies
    bool has_new;                                 // this position is the last key of the last block
    __device__ __forceinline__ PaHead(const PaArgs& a, uint32_t head, uint32_t pos, uint32_t wave) {
        h = head; kvh = head / (a.heads / a.kv_heads);
        const uint32_t seq = pos + 1;
        b = wave; nb = (seq + PA_B - 1) / PA_B; bs = b * PA_B;
        bl = b < AW && bs < seq ? min(PA_B, seq - bs) : 0u;
        has_new = b < AW && bs <= pos && pos < bs + PA_B;
        nk = has_new ? bl - 1 : bl;
        delta = pa_sgpr(bl ? pa_row(a, bs) - bs : 0u);
        zero = pa_sgpr(pa_row(a, 0));
    }
    __device__ __forceinline__ void load(PaKv<HD>& kv, const PaArgs& a, const PaLayer& L, uint32_t pos, uint32_t lane) const {
        if (!bl) return;
        const uint16_t* kb = pa_lds_ptr(L.kc) + kvh * HD;
        const uint32_t row = bs + lane, at = (row < pos ? row + delta : zero) * a.KV * 2;      // lanes without a cached key: the first row
        uint4 kr[HD / 8];
#pragma unroll
        for (int c = 0; c < HD / 8; c++) kr[c] = pa_at<uint4>(kb, at + c * 16);
        PaRaw<HD> raw;
        pa_load_values<HD>(raw, pa_lds_ptr(L.vc) + kvh * HD, bs, pos, delta, zero, a.KV, lane);
        pa_pack_values<HD>(kv, raw);
        kv.set_keys(kr);
    }
    template <bool SUMS>
    __device__ __forceinline__ void step(PaKv<HD>& kv, const PaArgs& a, const PaLayer& L, PaAttn<HD, AW>* sh, const uint64_t* exp_tab, uint32_t pos, uint32_t tag_in, PollCtx& cx) const;
};

template <int HD, uint32_t AW>
template <bool SUMS>
__device__ __forceinline__ void PaHead<HD, AW>::step(PaKv<HD>& kv, const PaArgs& a, const PaLayer& L, PaAttn<HD, AW>* sh, const uint64_t* exp_tab, uint32_t pos, uint32_t tag_in,
                                                     PollCtx& cx) const {
        constexpr int DPL = PaKv<HD>::DPL, KC = PaKv<HD>::KC;
        const uint32_t kv_stride = a.KV, lane = cx.lane;
        const float scale = 1.0f / sqrtf((float)HD);
        const PaExpTab tab{exp_tab};
        // the score of this position and the blocks' exp_scale are the work of waves without a block, as long as there are such
        const bool wave_new = b == nb % AW, wave_es = nb > 1 && b == (nb + 1) % AW;
        const uint16_t* vb = pa_lds_ptr(L.vc) + kvh * HD;
        uint32_t nk = pa_sgpr(this->nk);
        asm volatile("" : "+s"(nk));              // conditions on it are formed where they are used: kept from layer to layer they would not fit the registers
        if (cx.tid < pa_up(HD, 64)) {
            uint32_t g[3];
            const uint32_t e = min(cx.tid, (uint32_t)HD - 1);
            poll_tagged<3>([&](int i) { return i == 0 ? a.tq + (size_t)h * HD + e : a.tkv + (i == 1 ? 0u : a.KV) + kvh * HD + e; }, [&](int) { return tag_in; }, g, cx);
            if (cx.tid < HD) {
                sh->q[e] = __uint_as_float(g[0]);
                sh->pn[e] = __uint_as_float(g[0]) * f16_bits_to_f32((uint16_t)g[1]);
                sh->vn[e] = f16_bits_to_f32((uint16_t)g[2]);
            }
        }
        __syncthreads();
        if (*cx.sh_abort) return;
        float sc = -INFINITY;
        if (bl) {
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < HD; i++) {
                if (i % 16 == 0) __builtin_amdgcn_sched_barrier(0);      // all of q at once would not fit the registers
                sum = sum + sh->q[i] * kv.key(i);
            }
            if (lane < nk) sc = sum * scale;
            const float mb = wave_max(sc);
            if (lane == 0) sh->bmax[b] = mb;
        }
        if (wave_new) {
            float sum = 0.f;
#pragma unroll
            for (int i = 0; i < HD; i++) {
                if (i % 32 == 0) __builtin_amdgcn_sched_barrier(0);
                sum = sum + sh->pn[i];
            }
            if (lane == 0) sh->snew = sum * scale;
        }
        __syncthreads();
        if (wave_es) {
            // m after block i: the largest block maximum so far; es[0] = exp(-inf - m) is 0
            float m = -INFINITY, before = -INFINITY;
#pragma unroll
            for (uint32_t i = 0; i < AW; i++) {
                const float v = i < nb ? (i == nb - 1 ? fmaxf(sh->bmax[i], sh->snew) : sh->bmax[i]) : -INFINITY;
                if (i < lane) before = fmaxf(before, v);
                if (i <= lane) m = fmaxf(m, v);
            }
            const float es = expf_ref_with<true>(before - m, tab);
            if (lane < nb) sh->es[lane] = es;
        }
        if (bl) {
            float m = wave_max(lane <= b ? sh->bmax[lane] : -INFINITY);
            if (has_new) {
                const float s = sh->snew;
                m = fmaxf(m, s);
                if (lane == nk) sc = s;
            }
            sh->e[b][lane] = lane < bl ? expf_ref_with<true>(sc - m, tab) : 0.f;       // LDS operations of one wave execute in order
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
            float l_block = 0.f, sum[DPL];
#pragma unroll
            for (int t = 0; t < DPL; t++) sum[t] = 0.f;
#pragma nounroll
            for (uint32_t k0 = 0; k0 < PA_B; k0 += KC) {
                if (k0 && k0 >= nk) break;
                if (k0) { PaRaw<HD> raw; pa_load_values<HD>(raw, vb, bs + k0, pos, delta, zero, kv_stride, lane); pa_pack_values<HD>(kv, raw); }
                // keys past the last one are left out, not given a weight of 0: 0 * v is not 0 for an infinite v
#pragma unroll
                for (int i16 = 0; i16 < KC; i16 += 16) {
                    __builtin_amdgcn_sched_barrier(0);       // all weights at once would not fit the registers
                    if (k0 + i16 < nk) {
                        float w[16];
#pragma unroll
                        for (int i = 0; i < 16; i += 4) *reinterpret_cast<float4*>(w + i) = *reinterpret_cast<const float4*>(&sh->e[b][k0 + i16 + i]);
                        auto add = [&](int i) {
                            l_block = l_block + w[i];
#pragma unroll
                            for (int t = 0; t < DPL; t++) sum[t] = sum[t] + w[i] * kv.value(i16 + i, t);
                        };
                        if (k0 + i16 + 16 <= nk) {
#pragma unroll
                            for (int i = 0; i < 16; i++) add(i);
                        } else {
#pragma unroll
                            for (int i = 0; i < 16; i++)
                                if (k0 + i16 + i < nk) add(i);
                        }
                    }
                }
            }
            if (has_new) {
                const float w = sh->e[b][nk];
                l_block = l_block + w;
#pragma unroll
                for (int t = 0; t < DPL; t++) sum[t] = sum[t] + w * sh->vn[min(lane + 64 * t, (uint32_t)HD - 1)];
            }
#pragma unroll
            for (int t = 0; t < DPL; t++)
                if (lane + 64 * t < HD) sh->sums[b][lane + 64 * t] = sum[t];
            if (lane == 0) sh->lblk[b] = l_block;
        }
        __syncthreads();
        if (cx.tid < pa_up(HD, 64)) {
            const uint32_t d = cx.tid < HD ? cx.tid : 0;
            float l_i = 0.f + sh->lblk[0], acc = 0.f + sh->sums[0][d];               // es[0] = 0 times 0, then the sum
            for (uint32_t i = 1; i < nb; i++) {
                const float exp_scale = sh->es[i];
                l_i = l_i * exp_scale;
                acc = acc * exp_scale;
                l_i = l_i + sh->lblk[i];
                acc = acc + sh->sums[i][d];
            }
            const float inv_l = 1.0f / l_i;
            const float o = acc * inv_l;
            const uint32_t e = h * HD + cx.tid;
            pa_store_block<SUMS>(cx.tid < HD ? o : 0.f, a.taq + e / 32 * 9, tag_in + 1, cx.lane, cx.tid < HD);
        }
}

// Longer contexts where the order is free, a kernel of their own (beside the short form's registers neither has enough: 957 us a token at 2400 rows of the 1B
// shape, 483 apart): workgroup (KV head, split) attends to its part of the keys, a fetching wave per query head of the group (and the next four heads behind
// these); a head's workgroup merges the splits.  A pass is 8 keys (heads of 64; 4 of wider ones), 16 bytes of K and V a lane; a split's first PA_PASSES are
// requested before the workgroup waits for the query, further rounds of them when those are done.
constexpr int PA_PASSES = 10;
constexpr uint32_t PA_SPLITS = 32, PA_LDS = 64000, PA_ROUNDS = 8;
constexpr uint32_t PA_PAGES = PA_ROUNDS * PA_PASSES * 8 / PA_B + 2;       // pages that a split's rows lie in
template <int HD>
struct PaPart {
    static constexpr int LPK = HD <= 64 ? 8 : 16, KPW = 64 / LPK, REC = HD + 2;
    uint32_t kvh, split, t0, t1, zero;        // keys [t0, t1); where the first row lies
    bool on;
    __device__ __forceinline__ PaPart(const PaArgs& a, uint32_t wg, uint32_t pos) {
        kvh = wg % a.kv_heads; split = wg / a.kv_heads;
        const uint32_t seq = pos + 1, chunk = pa_up((seq + a.splits - 1) / max(a.splits, 1u), KPW);
        on = split < a.splits;
        t0 = min(split * chunk, seq);
        t1 = min(t0 + chunk, seq);
        zero = pa_sgpr(pa_row(a, 0));
    }
    // pages: the pool pages from t0's on, in LDS; rows that are not cached or another split's: the first row
    __device__ __forceinline__ void load(Half8* k, Half8* v, const PaArgs& a, const PaLayer& L, uint32_t from, const uint32_t* pages, uint32_t pos, uint32_t lane) const {
        const uint16_t* kc = pa_lds_ptr(L.kc) + kvh * HD;
        const uint16_t* vc = pa_lds_ptr(L.vc) + kvh * HD;
        const uint32_t c = min(lane % LPK, (uint32_t)HD / 8 - 1);
#pragma unroll
        for (int p = 0; p < PA_PASSES; p++) {
            const uint32_t t = from + p * KPW + lane / LPK;
            uint32_t row = t;
            if (a.pages) row = (pages[min((t >> a.page_shift) - (t0 >> a.page_shift), PA_PAGES - 1)] << a.page_shift) + (t & ((1u << a.page_shift) - 1u));
            const uint32_t at = ((t < min(t1, pos) ? row : zero) * a.KV + c * 8) * 2;
            k[p] = pa_at<Half8>(kc, at);
            v[p] = pa_at<Half8>(vc, at);
        }
    }
    // q_s: the group's heads in LDS, new_s: this position's K row and V row, fp16 pairs.  After the barrier that publishes them.
    __device__ __forceinline__ void attend(Half8* k, Half8* v, const PaArgs& a, const PaLayer& L, const float* q_s, const Half8* new_s, const uint32_t* pages, uint32_t pos, uint32_t tag_out,
                                           const PollCtx& cx) const {
        const uint32_t gsize = a.heads / a.kv_heads, lane = cx.lane, slot = lane / LPK, c = lane % LPK;
        const bool dvalid = c * 8 < (uint32_t)HD;
        const float scale = 1.0f / sqrtf((float)HD);
        const uint32_t cv = min(c, (uint32_t)HD / 8 - 1);
        uint32_t nk[4], nv[4];
#pragma unroll
        for (int i = 0; i < 4; i++) { nk[i] = new_s[cv].w[i]; nv[i] = new_s[HD / 8 + cv].w[i]; }
        for (uint32_t g = cx.wave; g < gsize; g += PA_POLL) {
            float qf[8], acc[8], m = -INFINITY, l = 0.f;
#pragma unroll
            for (int i = 0; i < 8; i++) { qf[i] = dvalid ? q_s[g * HD + c * 8 + i] : 0.f; acc[i] = 0.f; }
            for (uint32_t from = t0; from < t1; from += PA_PASSES * KPW) {
                if (from != t0 || g >= PA_POLL) load(k, v, a, L, from, pages, pos, lane);
#pragma unroll
                for (int p0 = 0; p0 < PA_PASSES; p0 += 2) {
                    const uint32_t tp = from + p0 * KPW;
                    if (tp < t1) {
                        float sc[2];
                        Half8 vv[2];
#pragma unroll
                        for (int u = 0; u < 2; u++) {
                            const uint32_t t = tp + u * KPW + slot;
                            Half8 kk;
                            // what is read in place of a key that is not there, or past a row's end, counts as 0: a weight of 0 times an infinite value would not
#pragma unroll
                            for (int i = 0; i < 4; i++) {
                                kk.w[i] = !dvalid ? 0u : t == pos ? nk[i] : k[p0 + u].w[i];
                                vv[u].w[i] = t >= t1 ? 0u : t == pos ? nv[i] : v[p0 + u].w[i];
                            }
                            const float d = key_dot<LPK>(qf, kk);
                            sc[u] = t < t1 ? d * scale : -INFINITY;
                        }
                        softmax_block_update<2>(m, l, acc, sc, vv);
                    }
                }
            }
            // fold the key slots: every lane of a column ends with the same sums
            auto fold = [&](auto O) {
                const float m2 = lane_xor<O.value>(m), l2 = lane_xor<O.value>(l), mn = fmaxf(m, m2);
                const float s1 = m == -INFINITY ? 0.f : __expf(m - mn), s2 = m2 == -INFINITY ? 0.f : __expf(m2 - mn);
                l = l * s1 + l2 * s2;
#pragma unroll
                for (int i = 0; i < 8; i++) acc[i] = acc[i] * s1 + lane_xor<O.value>(acc[i]) * s2;
                m = mn;
            };
            if (LPK == 8) fold(std::integral_constant<int, 8>{});
            fold(std::integral_constant<int, 16>{});
            fold(std::integral_constant<int, 32>{});
            uint64_t* rec = a.trec + ((size_t)(kvh * gsize + g) * a.splits + split) * REC;
#pragma unroll
            for (int j = 0; j < 8 / KPW; j++) {               // lane (slot, column): element column 8 + slot + KPW j
                float x = acc[KPW * j];
#pragma unroll
                for (int i = 1; i < KPW; i++) x = slot == (uint32_t)i ? acc[KPW * j + i] : x;
                if (dvalid) stc64(rec + c * 8 + slot + KPW * j, tag_out, __float_as_uint(x));
            }
            if (lane < 2) stc64(rec + HD + lane, tag_out, __float_as_uint(lane ? l : m));
        }
    }
};

// The splits of head h into its quantised row; recs: splits records, wt: a weight per split.  Fetching waves; two barriers.
template <int HD, bool SUMS>
__device__ __forceinline__ void pa_merge(const PaArgs& a, uint32_t h, uint32_t tag_in, uint32_t tag_out, float* recs, float* wt, const PollCtx& cx) {
    constexpr uint32_t REC = HD + 2, N = (PA_SPLITS * REC + PA_POLL_THREADS - 1) / PA_POLL_THREADS;
    const uint32_t ne = a.splits * REC;
    const uint64_t* base = a.trec + (size_t)h * ne;
    uint32_t v[N];
    poll_tagged<N>([&](int i) { return base + min(cx.tid + i * PA_POLL_THREADS, ne - 1); }, [&](int) { return tag_in; }, v, cx);
#pragma unroll
    for (uint32_t i = 0; i < N; i++)
        if (cx.tid + i * PA_POLL_THREADS < ne) recs[cx.tid + i * PA_POLL_THREADS] = __uint_as_float(v[i]);
    __syncthreads();
    if (*cx.sh_abort) return;
    if (cx.wave == 0) {
        const bool in = cx.lane < a.splits;
        const float m = in ? recs[cx.lane * REC + HD] : -INFINITY, l = in ? recs[cx.lane * REC + HD + 1] : 0.f;
        const float mx = wave_max(m);
        const float w = m == -INFINITY ? 0.f : __expf(m - mx);
        const float den = wave_sum(w * l);
        if (in) wt[cx.lane] = w / den;
    }
    __syncthreads();
    if (cx.tid < pa_up(HD, 64)) {
        const uint32_t d = min(cx.tid, (uint32_t)HD - 1);
        float o = 0.f;
#pragma unroll 8
        for (uint32_t i = 0; i < a.splits; i++) o = fmaf(wt[i], recs[i * REC + d], o);
        const uint32_t e = h * HD + cx.tid;
        pa_store_block<SUMS>(cx.tid < HD ? o : 0.f, a.taq + e / 32 * 9, tag_out, cx.lane, cx.tid < HD);
    }
}

// The tag of a phase instance: tag_base + 6 layer + 1 q;k;v, 2 attention (long contexts: its parts, 3 their merge), 4 o, 5 gate;up, 6 down; the argmax's is behind
// the last layer's.
template <typename F, bool ORD, bool LONG, int HD, PaFmt W, PaFmt LMW>
__global__ __launch_bounds__(PA_THREADS) void decode_ahead_kernel(PaArgs a) {
    constexpr bool SUMS = W == PA_KQ;
    static_assert(!SUMS || (!ORD && LMW == PA_KQ), "models of K-quant matrices: all of them, where the order is free");
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ uint32_t sh_abort;
    __shared__ ArgPair sh_arg[PA_WAVES];
    __shared__ float norm_part[PA_POLL];
    __shared__ uint32_t sh_pages[LONG ? PA_PAGES : 1];
    __shared__ uint64_t exp_tab[32];          // expf_ref's table
    uint32_t* aq = reinterpret_cast<uint32_t*>(smem);
    float* as = reinterpret_cast<float*>(smem + a.off_as);
    float* code_sums = reinterpret_cast<float*>(smem + a.off_as + a.to_sums);
    float* xs = reinterpret_cast<float*>(smem + a.off_xs);
    float* out = reinterpret_cast<float*>(smem + a.off_out);                     // the workgroup's row sums
    float* silu = reinterpret_cast<float*>(smem + a.off_silu);
    const PaLayer* layers = reinterpret_cast<const PaLayer*>(smem + a.off_layers);
    auto* attn = reinterpret_cast<PaAttn<HD, F::AW>*>(smem + a.off_attn);

    PollCtx cx;
    cx.tid = threadIdx.x;
    cx.lane = threadIdx.x & 63u;
    cx.wave = pa_sgpr(threadIdx.x >> 6);
    cx.wg = blockIdx.x;
    cx.G = a.G;
    cx.spin_limit = a.spin_limit;
    cx.sh_abort = &sh_abort;
    cx.abort_flag = a.state + 3;
    const bool comp = cx.wave >= PA_POLL;
    const uint32_t c = comp ? cx.wave - PA_POLL : 0u;
    if (cx.tid == 0) sh_abort = 0;
    if (cx.tid < 32) exp_tab[cx.tid] = expf_detail::tab((int)cx.tid);
    for (uint32_t i = cx.tid; i < a.lds_words; i += PA_THREADS) reinterpret_cast<uint32_t*>(smem)[i] = 0;      // the zeros behind products and accumulators
    for (uint32_t i = cx.tid; i < (a.L + 1) * (uint32_t)(sizeof(PaLayer) / 4); i += PA_THREADS)
        reinterpret_cast<uint32_t*>(smem + a.off_layers)[i] = ldg(reinterpret_cast<const uint32_t*>(a.layers) + i);
    const uint32_t pos = pa_sgpr(a.state[0]);
    const float* emb = a.embed + (size_t)a.token * a.H;
    if constexpr (LONG) {
        if (a.pages && cx.tid < PA_PAGES) sh_pages[cx.tid] = ldg(a.pages + min((PaPart<HD>(a, cx.wg, pos).t0 >> a.page_shift) + cx.tid, a.n_pages - 1));
    }
    __syncthreads();

    const uint32_t ntid = cx.tid - PA_POLL_THREADS;                               // of a computing thread
    // A phase ends, and the next one begins, where the first workgroup with a part of it has handed that on: a wait for the others' parts is the next phase's.
    auto stamp = [&](uint32_t wg, uint32_t slot, uint32_t slots = 1) {
        if (a.stamps && cx.wg == wg && cx.tid == 0) {
            const unsigned long long t = wall_clock64();
            for (uint32_t i = 0; i < slots; i++) a.stamps[slot + i] = t;
        }
    };
    PaSet<F::UL, LMW> wl[2];
    float4 n1;                                // norm weights of elements 4 ntid ..
    const PaMat ml = a.m[4];
    const uint32_t T = gridDim.x, WAVES = PA_COMP * T, lwv = c * T + cx.wg;
    auto load_norm = [&](const float* nw) { return pa_at<float4>(nw, min(ntid * 4, a.H - 4) * 4); };      // threads past the last one: it again
    // the barriers and what lies between them from a fetched row to its codes, for fetching and computing waves; false: the step is given up
    auto norm_fetching = [&]() {
        __syncthreads();
        if (sh_abort) return false;
        if (ORD) { pa_norm_sum(xs, a.xstride, a.eps, a.H, norm_part, cx); __syncthreads(); }
        __syncthreads();
        return true;
    };
    // Wide: where weights would be requested while others wait for a hand-over, the workgroup waits for an element of it too (requested at once they fill the memory
    // system in front of it: 545 us a token at the 1B shape, 451 so)
    // (a workgroup on which nothing depends may come late and find a later phase's element there)
    auto glance = [&](const uint64_t* p, uint32_t tag) {
        if (cx.wave == 0) poll_tagged<1, true>([&](int) { return p; }, [&](int) { return tag; }, nullptr, cx);
        __syncthreads();
        return sh_abort == 0;
    };
    auto norm_computing = [&](float4 n) {
        __syncthreads();
        if (sh_abort) return false;
        if (ORD) __syncthreads();
        pa_norm_quant<ORD, SUMS>(xs, a.xstride, n, a.eps, a.H, smem, a.off_as, a.to_sums, norm_part, ntid);
        __syncthreads();
        return true;
    };
    const uint32_t pos_row = pa_sgpr(pa_row(a, pos));
    const uint32_t head = cx.wg - a.head0;
    const bool on_a = head < a.heads;         // unsigned

    if (cx.wg < cx.G) {
        const PaMat mq = a.m[0], mo = a.m[1], mg = a.m[2], md = a.m[3];
        const uint32_t per_wave = 32 / PA_COMP;                                  // gate;up: 4 gate and 4 up rows a wave
        // a workgroup's rows lie side by side: one store hands them over
        auto rank = [&](const PaMat& m) { return cx.wg >= m.wg0 && (!F::WIDE || !on_a || &m == &md) ? cx.wg - m.wg0 : 0xFFFFFFu; };
        const uint32_t kq = rank(mq), ko = rank(mo), kd = rank(md);
        const uint32_t row_q = kq * PA_COMP * mq.R, row_o = ko * PA_COMP * mo.R, row_d = kd * PA_COMP * md.R;
        const bool on_q = row_q < mq.N, on_o = row_o < mo.N, on_g = cx.wg < a.I / 32, on_d = row_d < md.N;
        const PaTask tq = pa_task(mq, kq * PA_COMP + c, (kq * PA_COMP + c) * mq.R < a.QKS + a.KV ? a.six[0] : a.six_v), to = pa_task(mo, ko * PA_COMP + c, a.six[1]),
                     td = pa_task(md, kd * PA_COMP + c, a.six[3]);
        const PaTask tg{on_g ? (cx.wg * 32 + c * per_wave) * mg.nblk : 0u, on_g ? 2 * per_wave * mg.nblk : 0u, per_wave * mg.nblk, (a.I - per_wave) * mg.nblk, a.six[2]};
        const uint32_t pq = mq.prod + c * a.prod_words * 4, po = mo.prod + c * a.prod_words * 4, pg = mg.prod + c * a.prod_words * 4, pd = md.prod + c * a.prod_words * 4;
        // the first wave finishes rows: lane r the workgroup's r-th
        float rc = 1.f, rs = 0.f;                                                // rotation of its row of q | k
        const uint32_t qrow = row_q + cx.lane;
        const bool mine_q = cx.wave == 0 && cx.lane < PA_COMP * mq.R && qrow < mq.N;
        if (mine_q && qrow < a.QKS + a.KV) {
            const uint32_t d = (qrow < a.QKS ? qrow : qrow - a.QKS) % HD;
            rc = ldg(a.cos_t + (size_t)pos * (HD / 2) + d / 2);
            rs = ldg(a.sin_t + (size_t)pos * (HD / 2) + d / 2);
        }
        // Fetching and computing waves go through the layers in loops of their own (with the same barriers): neither keeps the other's registers.
        if (!comp) {
            const PaHead<HD, F::AW> ph(a, F::WIDE && on_a ? head : 0u, pos, cx.wave);
            const PaPart<HD> part(a, cx.wg, pos);
            float* q_s = reinterpret_cast<float*>(attn);                         // long contexts: the group's heads, then this position's K and V row
            Half8* new_s = reinterpret_cast<Half8*>(q_s + a.heads / a.kv_heads * HD);
#pragma nounroll
            for (uint32_t l = 0; l < a.L; l++) {
                // The thread's number is read afresh in every layer: addresses that follow from it would be kept from layer to layer and not fit the registers.
                asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
                const PaLayer& L = layers[l];
                const uint32_t base = a.tag_base + 6 * l, x_in = l ? base : 0u;
                // ---- norm | q;k;v | rotation, cache row
                stamp(0, 6 * l);
                Half8 pk[LONG ? PA_PASSES : 1], pv[LONG ? PA_PASSES : 1];
                if constexpr (LONG) {
                    if (part.on && cx.wave < a.heads / a.kv_heads) part.load(pk, pv, a, L, part.t0, sh_pages, pos, cx.lane);
                }
                if (on_q) {
                    uint16_t* kc = pa_lds_ptr(L.kc);
                    uint16_t* vc = pa_lds_ptr(L.vc);
                    pa_fetch_x<F::NX, ORD>(a.tx, x_in, emb, a.H, xs, a.xstride, norm_part, cx);
                    if (!norm_fetching()) return;
                    __syncthreads();
                    if (cx.wave == 0) {
                        const float v = out[cx.lane];
                        const float other = lane_xor<1>(v);                      // rope (emit.rs:508-528): rows 2i, 2i + 1 of a head
                        const float o = (qrow & 1u) ? other * rs + v * rc : v * rc - other * rs;
                        const bool is_q = qrow < a.QKS, is_k = qrow < a.QKS + a.KV;
                        const uint16_t hb = f32_to_f16_bits(is_k ? o : v);
                        const uint32_t at = qrow - a.QKS;                        // of [K row | V row]
                        if (mine_q) {
                            stc64(is_q ? a.tq + qrow : a.tkv + at, base + 1, is_q ? __float_as_uint(o) : (uint32_t)hb);
                            if (!is_q) stg((is_k ? kc + at : vc + (at - a.KV)) + (size_t)pos_row * a.KV, hb);
                        }
                    }
                }
                // ---- attention
                stamp(0, 6 * l + 1);
                if constexpr (LONG) {
                    if (part.on) {
                        // the group's heads, this position's K row and V row
                        const uint32_t gsize = a.heads / a.kv_heads, nq = gsize * HD, ne = nq + 2 * HD;
                        constexpr int N = 4;
                        uint32_t v[N];
                        auto at = [&](uint32_t e) {
                            e = min(e, ne - 1);
                            return e < nq ? a.tq + (size_t)part.kvh * nq + e : a.tkv + (e - nq < HD ? part.kvh * HD + (e - nq) : a.KV + part.kvh * HD + (e - nq - HD));
                        };
                        poll_tagged<N>([&](int i) { return at(cx.tid + i * PA_POLL_THREADS); }, [&](int) { return base + 1; }, v, cx);
#pragma unroll
                        for (int i = 0; i < N; i++) {
                            const uint32_t e = cx.tid + i * PA_POLL_THREADS;
                            if (e < nq) q_s[e] = __uint_as_float(v[i]);
                            else if (e < ne) reinterpret_cast<uint16_t*>(new_s)[e - nq] = (uint16_t)v[i];
                        }
                        __syncthreads();
                        if (sh_abort) return;
                        part.attend(pk, pv, a, L, q_s, new_s, sh_pages, pos, base + 2, cx);
                        stamp(0, 6 * l + 2);
                    } else if (!glance(a.tkv + 2 * a.KV - 1, base + 1)) {
                        return;
                    }
                    if (on_a) {
                        pa_merge<HD, SUMS>(a, head, base + 2, base + 3, reinterpret_cast<float*>(smem + a.off_rec), silu, cx);
                        if (sh_abort) return;
                        stamp(a.head0, 6 * l + 3);
                    } else if (!on_o && !glance(a.taq + a.QKS / 32 * 9 - 1, base + 3)) {
                        return;
                    }
                } else if constexpr (F::WIDE) {
                    if (on_a) {
                        PaKv<HD> kv;
                        ph.load(kv, a, L, pos, cx.lane);
                        ph.template step<SUMS>(kv, a, L, attn, exp_tab, pos, base + 1, cx);
                        stamp(a.head0, 6 * l + 2, 2);                            // no merge phase
                    } else {
                        if (!glance(a.tkv + 2 * a.KV - 1, base + 1)) return;
                    }
                    if (sh_abort) return;
                    if (!on_o && !on_a && !glance(a.taq + a.QKS / 32 * 9 - 1, base + 2)) return;
                }
                // ---- o + residual
                if (on_o) {
                    const bool mine = cx.wave == 0 && cx.lane < PA_COMP * mo.R && row_o + cx.lane < mo.N;
                    const float r = pa_fetch_aq<F::NV, SUMS>(a.taq, base + (LONG ? 3 : 2), a.QKS, aq, as, code_sums, mine, row_o + cx.lane, a.tx, x_in, emb, cx);
                    __syncthreads();
                    if (sh_abort) return;
                    __syncthreads();
                    if (mine) stc64(a.tx + row_o + cx.lane, base + 4, __float_as_uint(r + out[cx.lane]));     // residual_add, emit.rs:455-459
                }
                // ---- norm | gate;up | silu(gate) * up
                stamp(mo.wg0, 6 * l + 4);
                if (on_g) {
                    pa_fetch_x<F::NX, ORD>(a.tx, base + 4, emb, a.H, xs, a.xstride, norm_part, cx);
                    if (!norm_fetching()) return;
                    __syncthreads();
                    if (cx.wave == 0) pa_store_block<SUMS>(silu[cx.lane & 31u], a.taq2 + cx.wg * 9, base + 5, cx.lane, cx.lane < 32);
                }
                // ---- down + residual
                stamp(0, 6 * l + 5);
                if (on_d) {
                    const bool mine = cx.wave == 0 && cx.lane < PA_COMP * md.R && row_d + cx.lane < md.N;
                    const float r = pa_fetch_aq<F::NV, SUMS>(a.taq2, base + 5, a.I, aq, as, code_sums, mine, row_d + cx.lane, a.tx, base + 4, emb, cx);
                    __syncthreads();
                    if (sh_abort) return;
                    __syncthreads();
                    if (mine) stc64(a.tx + row_d + cx.lane, base + 6, __float_as_uint(r + out[cx.lane]));
                }
            }
        } else {
            PaSet<F::UQ, W> wq;
            PaSet<F::UO, W> wo;
            PaSet<F::UG1, W> wg;
            PaSet<F::WIDE ? F::UG2 : F::UD, W> wd;                              // Wide: first gate;up's second part, then (unless EARLY) down
            // EARLY: down's weights take the place of gate;up's first part, half of them requested ahead of the second part's products and half behind: the memory has work
            // while a workgroup computes, and what the result's store and the next poll wait behind is on its way by then.  (All of down behind the results' barrier / this, 1B
            // shape, us a token by rows of context: Q8_0 33 430 / 400, 300 463 / 440, 2400 477 / 457, order-faithful 33 471 / 450; Q4_K and Q6_K 33 487 / 457, 2400 539 / 511;
            // 8 layers of 1024 channels Q8_0 151 / 151, of 1280 163 / 160.  All of down ahead of the second part's products 472 for the first of these, none of it 412, its second
            // half behind the row sums' barrier 418.)  Not Q4_0, half the bytes to wait for: 403 / 386 there,
            // but models of 1024 channels 150 / 153; one form for all its sizes, the one that costs none of them.  The other sets gain little or
            // nothing from an earlier place: q;k;v ahead of down's products 1 % (1024 channels 2 % slower), gate;up's second part ahead of o's products 2 to 6 us slower.
            constexpr bool EARLY = F::WIDE && W != PA_Q4;
            static_assert(!EARLY || F::UG1 == F::UD, "down takes the place of gate;up's first part");
            constexpr int HALF = F::UD / 2;
            float4 n2;
            n1 = load_norm(pa_lds_ptr(layers[0].norm[0]));
            pa_load(wq, pa_lds_ptr(layers[0].w[0]), tq, cx.lane);
            if (F::WIDE && on_a) pa_load(wg, pa_lds_ptr(layers[0].w[2]), tg, cx.lane);
#pragma nounroll
            for (uint32_t l = 0; l < a.L; l++) {
                asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
                const PaLayer& L = layers[l];
                const PaLayer& N = layers[l + 1];
                if (on_q) {
                    const auto x = pa_index<F::UQ, W>(tq, mq, a.off_as, pq, cx.lane);
                    if (!norm_computing(n1)) return;
                    pa_products(wq, x, tq, smem, a.to_sums);
                    const PaSum v = pa_row_sum<ORD>(mq, mq.R, smem + pq, cx.lane);
                    if (v.on) out[c * mq.R + v.row] = v.v;
                    __syncthreads();
                }
                if constexpr (F::WIDE) {
                    __syncthreads();
                    if (sh_abort) return;
                    if (on_a) { __syncthreads(); if (LONG && sh_abort) return; __syncthreads(); }
                }
                // While the attention is at work nothing else is on its way to this workgroup: now the matrices that follow are requested (a load that
                // misses ahead of a poll holds the poll up, whichever wave it belongs to).
                n2 = load_norm(pa_lds_ptr(L.norm[1]));
                n1 = load_norm(pa_lds_ptr(N.norm[0]));
                pa_load(wo, pa_lds_ptr(L.w[1]), to, cx.lane);
                if constexpr (F::WIDE) {
                    if (!on_a) pa_load(wg, pa_lds_ptr(L.w[2]), tg, cx.lane);
                    if (!on_o) {
                        if (!on_a) { __syncthreads(); if (sh_abort) return; }
                        pa_load<F::UG1>(wd, pa_lds_ptr(L.w[2]), tg, cx.lane);
                    }
                } else {
                    pa_load(wg, pa_lds_ptr(L.w[2]), tg, cx.lane);
                    pa_load(wd, pa_lds_ptr(L.w[3]), td, cx.lane);
                    pa_load(wq, pa_lds_ptr(N.w[0]), tq, cx.lane);
                }
                if (on_o) {
                    const auto x = pa_index<F::UO, W>(to, mo, a.off_as, po, cx.lane);
                    __syncthreads();
                    if (sh_abort) return;
                    pa_products(wo, x, to, smem, a.to_sums);
                    const PaSum v = pa_row_sum<ORD>(mo, mo.R, smem + po, cx.lane);
                    if (v.on) out[c * mo.R + v.row] = v.v;
                    __syncthreads();
                    if constexpr (F::WIDE) pa_load<F::UG1>(wd, pa_lds_ptr(L.w[2]), tg, cx.lane);
                }
                if (on_g) {
                    const auto x = pa_index<F::UG1, W>(tg, mg, a.off_as, pg, cx.lane);
                    if (!norm_computing(n2)) return;
                    pa_products(wg, x, tg, smem, a.to_sums);
                    if constexpr (F::WIDE) {
                        if constexpr (EARLY) pa_load<0, 0, HALF>(wg, pa_lds_ptr(L.w[3]), td, cx.lane);
                        pa_products<F::UG1>(wd, pa_index<F::UG2, W, F::UG1>(tg, mg, a.off_as, pg, cx.lane), tg, smem, a.to_sums);
                        if constexpr (EARLY) pa_load<0, HALF>(wg, pa_lds_ptr(L.w[3]), td, cx.lane);
                    }
                    const PaSum v = pa_row_sum<ORD>(mg, 2 * per_wave, smem + pg, cx.lane);
                    const float up = ORD ? lane_xor<4>(v.v) : lane_xor<32>(v.v);           // row r + 4 of 8
                    if (v.on && v.row < per_wave) silu[c * per_wave + v.row] = (v.v / (1.0f + expf_ref_with<true>(-v.v, PaExpTab{exp_tab}))) * up;      // silu_mul, emit.rs:380-386
                    __syncthreads();
                } else if constexpr (EARLY) {
                    pa_load(wg, pa_lds_ptr(L.w[3]), td, cx.lane);
                }
                if constexpr (F::WIDE && !EARLY) pa_load(wd, pa_lds_ptr(L.w[3]), td, cx.lane);
                if (on_d) {
                    const auto x = pa_index<F::UD, W>(td, md, a.off_as, pd, cx.lane);
                    __syncthreads();
                    if (sh_abort) return;
                    if constexpr (EARLY) pa_products(wg, x, td, smem, a.to_sums);
                    else pa_products(wd, x, td, smem, a.to_sums);
                    const PaSum v = pa_row_sum<ORD>(md, md.R, smem + pd, cx.lane);
                    if (v.on) out[c * md.R + v.row] = v.v;
                    __syncthreads();
                }
                if constexpr (F::WIDE) {
                    pa_load(wq, pa_lds_ptr(N.w[0]), tq, cx.lane);
                    if (on_a) pa_load(wg, pa_lds_ptr(N.w[2]), tg, cx.lane);
                }
            }
            pa_load(wl[0], a.lm, pa_task(ml, lwv, a.six[4]), cx.lane);
        }
    } else {
        if (comp) n1 = load_norm(pa_lds_ptr(layers[a.L].norm[0]));
        if constexpr (!F::WIDE) {
            if (on_a) {
                const PaHead<HD, F::AW> ph(a, head, pos, cx.wave);
#pragma nounroll
                for (uint32_t l = 0; l < a.L; l++) {
                    asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
                    PaKv<HD> kv;
                    ph.load(kv, a, layers[l], pos, cx.lane);                     // requested as soon as the layer before is done
                    ph.template step<SUMS>(kv, a, layers[l], attn, exp_tab, pos, a.tag_base + 6 * l + 1, cx);
                    if (sh_abort) return;
                    stamp(a.head0, 6 * l + 2, 2);
                }
            }
        }
        if (comp) pa_load(wl[0], a.lm, pa_task(ml, lwv, a.six[4]), cx.lane);
        // a workgroup without rows in the layers looks for the final row now and then only
        if (cx.tid == 0) {
            uint32_t spins = 0;
            while ((uint32_t)(ldc64(a.tx + a.H - 1) >> 32) != a.tag_base + 6 * a.L && ++spins <= cx.spin_limit &&
                   ((spins & 255u) != 0 || __hip_atomic_load(cx.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0))
                __builtin_amdgcn_s_sleep(16);
        }
        __syncthreads();
    }

    // ---- final norm | lm_head | argmax
    asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
    stamp(0, 6 * a.L);
    ArgPair best{-INFINITY, 0};
    if (!comp) {
        pa_fetch_x<F::NX, ORD>(a.tx, a.tag_base + 6 * a.L, emb, a.H, xs, a.xstride, norm_part, cx);
        if (!norm_fetching()) return;
    } else {
        const uint32_t pl = ml.prod + c * a.prod_words * 4;
        if (!norm_computing(n1)) return;
        auto tile = [&](uint32_t t, const PaSet<F::UL, LMW>& w) {
            const PaTask task = pa_task(ml, t, a.six[4]);
            pa_products(w, pa_index<F::UL, LMW>(task, ml, a.off_as, pl, cx.lane), task, smem, a.to_sums);
            const PaSum sum = pa_row_sum<ORD>(ml, pa_rows(ml, t), smem + pl, cx.lane);
            const uint32_t row = t * ml.R + sum.row;
            float v = sum.v;
            if (sum.on) {
                stg(a.logits + row, v);
                // apply_repeat_penalty (project.rs:505-513) ahead of the argmax.  The lane that holds the row of the token being fed is the
                // only one in the grid to touch that counter: it adds this step's occurrence.
                if (a.penalty > 1.0f) {
                    const bool fed = row == a.token;
                    const uint32_t n = ldg(a.counts + row) + (fed ? 1u : 0u);
                    if (fed) { stg(a.counts + row, n); stg(a.state + 4, a.step_seq); }      // so that a step that gives up later can be undone
                    v = repeat_penalised(v, n, a.penalty);
                }
                best = arg_better(best, ArgPair{v, row});
            }
        };
        for (uint32_t t = lwv; t * ml.R < ml.N; t += 2 * WAVES) {
            const bool second = (t + WAVES) * ml.R < ml.N, third = (t + 2 * WAVES) * ml.R < ml.N;
            if (second) pa_load(wl[1], a.lm, pa_task(ml, t + WAVES, a.six[4]), cx.lane);
            tile(t, wl[0]);
            if (third) pa_load(wl[0], a.lm, pa_task(ml, t + 2 * WAVES, a.six[4]), cx.lane);
            if (second) tile(t + WAVES, wl[1]);
        }
    }
    const uint32_t th = a.tag_base + 6 * a.L + 1;
    best = best_of_workgroup<PA_WAVES>(best, sh_arg, cx);
    if (cx.tid == 0) {
        stc64(a.tpart + 2 * cx.wg, th, __float_as_uint(best.v));
        stc64(a.tpart + 2 * cx.wg + 1, th, best.i);
    }
    stamp(0, 6 * a.L + 1);
    if (cx.wg != 0) return;
    ArgPair p{-INFINITY, 0};
    for (uint32_t w = cx.tid; w < T; w += PA_THREADS) {
        uint32_t v[2];
        poll_tagged<2>([&](int i) { return a.tpart + 2 * w + (uint32_t)i; }, [&](int) { return th; }, v, cx);
        p = arg_better(p, ArgPair{__uint_as_float(v[0]), v[1]});
    }
    p = best_of_workgroup<PA_WAVES>(p, sh_arg, cx);
    if (sh_abort) return;
    if (cx.tid == 0) {
        a.state[2] = p.i;
        a.state[1] = p.i;
        a.state[0] = pos + 1;
        if (!(a.penalty > 1.0f)) a.counts[a.token] += 1;          // nobody read the counters in this launch
        stamp(0, 6 * a.L + 2);
        // the host may be spinning on this word instead of waiting for the stream
        if (a.host_out) __hip_atomic_store(a.host_out, ((unsigned long long)a.host_seq << 32) | p.i, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

template <typename F, bool ORD, bool LONG, int HD>
const void* pa_kernel_hd(PaFmt w, PaFmt lm) {
    if constexpr (F::WIDE && !ORD) {
        if (w == PA_KQ) return reinterpret_cast<const void*>(decode_ahead_kernel<F, ORD, LONG, HD, PA_KQ, PA_KQ>);
    }
    if (w == PA_Q4)
        return lm == PA_Q4 ? reinterpret_cast<const void*>(decode_ahead_kernel<F, ORD, LONG, HD, PA_Q4, PA_Q4>) : reinterpret_cast<const void*>(decode_ahead_kernel<F, ORD, LONG, HD, PA_Q4, PA_Q8>);
    return lm == PA_Q4 ? reinterpret_cast<const void*>(decode_ahead_kernel<F, ORD, LONG, HD, PA_Q8, PA_Q4>) : reinterpret_cast<const void*>(decode_ahead_kernel<F, ORD, LONG, HD, PA_Q8, PA_Q8>);
}

// What a form means for a shape.
struct PaForm { int units[5]; uint32_t nx, nv, aw; bool wide; const void* kernel; uint32_t attn_bytes; };
template <typename F, bool ORD, bool LONG>
const void* pa_kernel(uint32_t hd, PaFmt w, PaFmt lm) {
    return hd == 64 ? pa_kernel_hd<F, ORD, LONG, 64>(w, lm) : hd == 96 ? pa_kernel_hd<F, ORD, LONG, 96>(w, lm) : pa_kernel_hd<F, ORD, LONG, 128>(w, lm);
}
template <typename F, bool ORD>
PaForm pa_form(uint32_t hd, PaFmt w, PaFmt lm) {
    return PaForm{{F::UQ, F::UO, F::UG1 + F::UG2, F::UD, F::UL}, F::NX, F::NV, F::AW, F::WIDE,
                  pa_kernel<F, ORD, false>(hd, w, lm),
                  (uint32_t)(hd == 64 ? sizeof(PaAttn<64, F::AW>) : hd == 96 ? sizeof(PaAttn<96, F::AW>) : sizeof(PaAttn<128, F::AW>))};
}

// A K-quant matrix as PA_KQ blocks, from the planes gemv_kquant.hip keeps.  One thread per (row, block).
__global__ __launch_bounds__(256) void pa_repack_kernel(bool q6, const uint8_t* __restrict__ qs, const uint8_t* __restrict__ meta, uint32_t K, uint64_t total, uint8_t* __restrict__ codes,
                                                        uint32_t* __restrict__ words) {
    const uint64_t id = (uint64_t)blockIdx.x * 256 + threadIdx.x;       // n * nblk + b
    if (id >= total) return;
    const uint32_t nblk = K / 32;
    const uint64_t n = id / nblk;
    const uint32_t b = (uint32_t)(id % nblk), j = b & 7;
    const uint64_t super = n * (K / 256) + b / 8;
    uint8_t* dst = codes + id * 32;
    if (q6) {
        // block 4 h + r: r = 0, 1 the low nibbles of ql[64 h + 32 r ..], r = 2, 3 the high nibbles of ql[64 h + 32 (r - 2) ..]; bit pair r of qh[32 h ..]
        const uint8_t *sp = qs + super * 192, *mp = meta + super * 32;
        const uint32_t h = j >> 2, r = j & 3;
        const uint8_t *ql = sp + 64 * h + 32 * (r & 1), *qh = sp + 128 + 32 * h;
        for (uint32_t e = 0; e < 32; e++) dst[e] = (uint8_t)(int8_t)((int)(((ql[e] >> (r >> 1) * 4) & 15u) | (((qh[e] >> 2 * r) & 3u) << 4)) - 32);
        words[id] = (uint32_t)mp[16] | ((uint32_t)mp[17] << 8) | ((uint32_t)mp[2 * j] << 16) | ((uint32_t)mp[2 * j + 1] << 24);
    } else {
        const uint8_t *mp = meta + super * 16, *s12 = mp + 4;
        uint32_t sc, mn;                                                 // get_scale_min_k4, emit.rs:3013-3021
        if (j < 4) { sc = s12[j] & 63u; mn = s12[j + 4] & 63u; }
        else {
            sc = (s12[j + 4] & 0x0Fu) | ((s12[j - 4] >> 6) << 4);
            mn = (s12[j + 4] >> 4) | ((s12[j] >> 6) << 4);
        }
        const uint8_t* src = qs + super * 128 + 32 * (j >> 1);           // the low nibbles (j even) or the high ones
        for (uint32_t e = 0; e < 32; e++) dst[e] = (uint8_t)((src[e] >> (j & 1) * 4) & 15u);
        words[id] = ((uint32_t)mp[2 * (j & 1)] | ((uint32_t)mp[2 * (j & 1) + 1] << 8)) | (sc << 16) | (mn << 24);
    }
}
void pa_repack(const QWeight& w, uint8_t* codes, uint32_t* words) {
    const uint64_t total = (uint64_t)w.N * (w.K / 32);
    fh::launch(pa_repack_kernel, dim3((uint32_t)((total + 255) / 256)), 256, 0, nullptr, w.wdtype == FORGE_HIP_Q6_K, w.qs, reinterpret_cast<const uint8_t*>(w.scales), w.K, total, codes, words);
}

}  // namespace

struct PaState {
    PaArgs args{};
    std::vector<void*> owned;
    const void* kernel = nullptr;
    const void* kernel_long = nullptr;
    uint32_t grid = 0, lds = 0, n_stamps = 0, max_rows = 0, one_rows = 0;
    bool cooperative = false;
    uint64_t* tagged = nullptr;
    size_t tagged_bytes = 0;
    std::vector<unsigned long long> stamps_host;
    int wall_khz = 0;
    unsigned long long* host_out = nullptr;
    unsigned long long* host_out_dev = nullptr;
    uint32_t seq = 0;
    ~PaState() {
        for (void* p : owned) (void)hipFree(p);
        if (host_out) (void)hipHostFree(host_out);
    }
    template <typename T>
    T* dev(size_t n) {
        void* p = nullptr;
        if (hipMalloc(&p, n < 16 ? 16 : n) != hipSuccess) return nullptr;
        owned.push_back(p);
        return static_cast<T*>(p);
    }
};

void pa_destroy(PaState* st) { delete st; }

// Lanes without a key of their own read the cache's first row, which an empty cache does not have yet.  The last context: what the attention's registers hold.
bool pa_covers(const PaState* st, int64_t pos) { return st && pos >= 1 && pos < (int64_t)st->max_rows; }

int32_t pa_create(const forge_hip_config& c, const std::vector<PdLayerIn>& layers, const QWeight& lm_head, const float* embed, const float* final_norm,
                  const float* cos_t, const float* sin_t, float* logits, uint32_t* state, uint32_t* counts, PaState** out) {
    *out = nullptr;
    const uint32_t H = c.hidden, I = c.inter, hd = c.head_dim, QKS = c.heads * hd, KV = c.kv_heads * hd;
    if (c.sliding_window != 0 || layers.empty()) return FORGE_HIP_OK;
    const bool kq = layers[0].q != nullptr;
    if (kq != lm_head.kquant() || (!kq && !layers[0].qkv)) return FORGE_HIP_OK;
    if (hd != 64 && hd != 96 && hd != 128) return FORGE_HIP_OK;
    const bool q4 = c.wdtype == FORGE_HIP_Q4_0, lmq4 = c.lm_head_dtype == FORGE_HIP_Q4_0;
    if (H < 64 || I < 64 || QKS < 64 || !decode_ahead_offsets_fit(c.max_seq, KV, c.vocab, H, lmq4)) return FORGE_HIP_OK;
    const bool exact = (c.flags & FORGE_HIP_FLAG_EXACT) != 0;
    // Matrices of K-quants: the wide form where the order is free, formats that are the same in every layer.
    const PaFmt fw = kq ? PA_KQ : q4 ? PA_Q4 : PA_Q8, fl = kq ? PA_KQ : lmq4 ? PA_Q4 : PA_Q8;
    if (kq) {
        if (exact || H <= PaNarrow::NX * PA_POLL_THREADS) return FORGE_HIP_OK;
        for (const PdLayerIn& in : layers) {
            const QWeight *now[7] = {in.q, in.k, in.v, in.o, in.gate, in.up, in.down}, *first[7] = {layers[0].q, layers[0].q, layers[0].v, layers[0].o, layers[0].gate, layers[0].gate, layers[0].down};
            for (int i = 0; i < 7; i++)
                if (!now[i] || !now[i]->kquant() || now[i]->wdtype != first[i]->wdtype) return FORGE_HIP_OK;
        }
    }
    const PaForm f = H <= PaNarrow::NX * PA_POLL_THREADS ? pa_form<PaNarrow, true>(hd, fw, fl) : exact ? pa_form<PaWide, true>(hd, fw, fl) : pa_form<PaWide, false>(hd, fw, fl);
    // what the polling threads fetch at once
    if (H > f.nx * PA_POLL_THREADS || I / 32 * 9 > f.nv * PA_POLL_THREADS || QKS / 32 * 9 > f.nv * PA_POLL_THREADS) return FORGE_HIP_OK;
    // rows that the reference adds in its four-accumulator order (the last len % 4 of a chunk) are left to the other kernels
    if (H % 4 || I % 4 || QKS % 4 || KV % 4 || c.vocab % 4) return FORGE_HIP_OK;
    int dev = 0, coop = 0, cus = 0, khz = 0;
    FH_HIP(hipGetDevice(&dev));
    FH_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
    FH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    FH_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));

    std::unique_ptr<PaState> st(new PaState());
    st->cooperative = resident_cooperative();
    if (st->cooperative && !coop) return FORGE_HIP_OK;
    PaArgs& a = st->args;
    const uint32_t nq[5] = {QKS + 2 * KV, H, 2 * I, H, c.vocab}, kk[5] = {H, QKS, H, I, H};
    for (int i = 0; i < 5; i++) {
        PaMat& m = a.m[i];
        m.N = nq[i]; m.nblk = kk[i] / 32;
        m.magic = (uint32_t)(0x100000000ull / m.nblk) + 1u;
        m.R = 64u * f.units[i] / m.nblk;                             // the most a wave can hold
        if (i == 0) m.R = std::min(m.R & ~1u, PA_MAX_ROWS);        // a rotation's pair in one wave
        else if (i == 1 || i == 3) m.R = std::min(m.R, PA_MAX_ROWS);
        else if (i == 2) { if (m.R < 64 / PA_COMP) return FORGE_HIP_OK; m.R = 64 / PA_COMP; }
        else m.R = std::min(m.R, 32u);
        if (m.R == 0) return FORGE_HIP_OK;
    }
    // Narrow: the fewest workgroups that hold every row at the most per wave, gate;up by whole blocks of 32, then a workgroup per head, and what is left of the device
    // for the lm_head; as few rows per wave as that many workgroups allow.
    // Wide: every workgroup a block of gate;up and of down's rows; the last ones a head each in place of rows of q;k;v and o, which lie at either end of the others.
    uint32_t g = I / 32;
    for (int i : {0, 1, 3}) g = std::max(g, (a.m[i].N + a.m[i].R * PA_COMP - 1) / (a.m[i].R * PA_COMP));
    if (g + (f.wide ? 0u : c.heads) > (uint32_t)cus || c.heads >= (uint32_t)cus) return FORGE_HIP_OK;
    st->grid = (uint32_t)cus;
    a.G = f.wide ? st->grid : g;
    a.head0 = f.wide ? st->grid - c.heads : g;
    for (int i : {0, 1, 3}) {
        const uint32_t n = f.wide && i != 3 ? a.head0 : a.G;             // workgroups that may hold rows
        uint32_t r = (a.m[i].N + n * PA_COMP - 1) / (n * PA_COMP);
        if (i == 0) r = pa_up(r, 2);
        if (r > a.m[i].R) return FORGE_HIP_OK;
        a.m[i].R = r;
        a.m[i].wg0 = f.wide && i == 1 ? n - (a.m[i].N + r * PA_COMP - 1) / (r * PA_COMP) : 0u;
    }
    if (kq) {
        auto six = [](const QWeight* w) { return w->wdtype == FORGE_HIP_Q6_K ? 1u : 0u; };
        const PdLayerIn& in = layers[0];
        a.six[0] = six(in.q); a.six_v = six(in.v); a.six[1] = six(in.o); a.six[2] = six(in.gate); a.six[3] = six(in.down); a.six[4] = six(&lm_head);
        if (a.six[0] != a.six_v && (QKS + KV) % a.m[0].R) return FORGE_HIP_OK;      // a wave's rows are of one format
    }
    a.L = (uint32_t)layers.size(); a.H = H; a.I = I; a.QKS = QKS; a.KV = KV; a.heads = c.heads; a.kv_heads = c.kv_heads;
    a.eps = c.rms_eps;
    const uint32_t kmax = std::max(std::max(H, I), QKS);
    a.off_as = pa_up(kmax, 16);
    a.to_sums = kq ? pa_up(kmax / 32 * 4, 16) : 0u;
    a.off_xs = a.off_as + pa_up(kmax / 32 * 4, 16) + a.to_sums;
    auto odd16 = [](uint32_t words) { return words % 8 ? words : words + 4; };      // rows an odd number of 16-byte units apart spread over the banks
    a.xstride = odd16(pa_up(H / 16, PA_SSQ));
    a.off_out = a.off_xs + 16 * a.xstride * 4;
    a.off_silu = a.off_out + PA_COMP * PA_MAX_ROWS * 4;
    a.off_prod = a.off_silu + 32 * 4;
    a.prod_words = 0;
    for (int i = 0; i < 5; i++) {
        PaMat& m = a.m[i];
        m.stride = odd16(pa_up(m.nblk, PA_SUM));
        while ((m.R << (m.fold + 1)) <= 64) m.fold++;
        // matrices of one depth share an area: the zeros behind their rows are the same
        int same = 0;
        while (a.m[same].nblk != m.nblk) same++;
        uint32_t rows = 0;
        for (int k = i; same == i && k < 5; k++)
            if (a.m[k].nblk == m.nblk) rows = std::max(rows, a.m[k].R);
        if (same == i) {
            m.prod = a.off_prod + a.prod_words * 4;
            m.dump = rows * m.stride * 4;
            a.prod_words += rows * m.stride + 4;
        } else {
            m.prod = a.m[same].prod;
            m.dump = a.m[same].dump;
        }
    }
    a.off_layers = a.off_prod + PA_COMP * a.prod_words * 4;
    a.lds_words = a.off_layers / 4;
    a.off_attn = pa_up(a.off_layers + ((uint32_t)layers.size() + 1) * (uint32_t)sizeof(PaLayer), 16);
    st->lds = a.off_attn + f.attn_bytes;
    if (st->lds > PA_LDS) return FORGE_HIP_OK;
    st->kernel = f.kernel;
    st->one_rows = st->max_rows = f.aw * PA_B;
    // Long contexts: as many splits as there are workgroups and room for a head's records in LDS (the group's heads and this position's rows are in PaAttn's place)
    const uint32_t gsize = c.heads / c.kv_heads, rec_bytes = (hd + 2) * 4;
    if (f.wide && !exact && gsize * hd + 2 * hd <= 4 * PA_POLL_THREADS && (gsize * hd + hd) * 4 <= f.attn_bytes) {
        const uint32_t n = std::min(std::min(PA_SPLITS, a.G / c.kv_heads), (PA_LDS - st->lds) / rec_bytes);
        if (n >= 8) {
            a.splits = n;
            a.off_rec = st->lds;
            st->lds += n * rec_bytes;
            // Rounds.  With a second head a wave, a third round is no longer hidden (us per token, decode_persistent.hip / this: 12/2 heads of 128, 2540 rows 287 / 270,
            // 3500: 286 / 293; 14/2 of 64, 5000: 241 / 210, 10000: 256 / 261); with few KV heads that kernel has more workgroups for the context.  Otherwise this
            // one is ahead up to the eighth round (8 layers of the 1B shape, 5000: 325 / 245, 20000: 377 / 337; 16/4 heads of 96, 10000: 368 / 308), but with heads of 128 not
            // past the sixth (16/8, 7000: 274 / 261, 10000: 289 / 296; 16/16, 3500: 270 / 264, 5000: 286 / 295), and with fewer than 16 splits, whose contexts are short, not
            // past the fifth (8 splits of 12/4 heads of 128, 1000: 226 / 201, 2400: 237 / 258; of 16/4 heads of 96, 1000: 261 / 217, 2400: 276 / 284; 4 splits of the 1B
            // shape, 1000: 307 / 257, 2400: 311 / 321).  Below 8 splits (more than 32 KV heads, or no LDS for more) there is little context left to cover.
            // Where two rounds are the line, K-quants, whose streamed matrices are fewer bytes, take one (12/2 heads of 128, 8192 wide, 1000: 274 / 275, 2400: 286 / 307).
            const uint32_t rounds = gsize > PA_POLL || c.kv_heads < 4 ? (kq ? 1 : 2) : n < 16 ? 5 : hd > 96 ? 6 : PA_ROUNDS;
            st->max_rows = std::min(c.max_seq, n * rounds * PA_PASSES * (hd <= 64 ? 8u : 4u));
            st->kernel_long = pa_kernel<PaWide, false, true>(hd, fw, fl);
        }
    }
    int per_cu = 0;
    for (const void* k : {st->kernel, st->kernel_long})
        if (k && (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k, PA_THREADS, st->lds) != hipSuccess || per_cu < 1)) { (void)hipGetLastError(); return FORGE_HIP_OK; }

    std::vector<PaLayer> host(layers.size() + 1);
    memset(host.data(), 0, host.size() * sizeof(PaLayer));
    if (kq) {
        uint64_t blocks = (uint64_t)lm_head.N * (lm_head.K / 32);
        for (const PdLayerIn& in : layers)
            for (const QWeight* w : {in.q, in.k, in.v, in.o, in.gate, in.up, in.down}) blocks += (uint64_t)w->N * (w->K / 32);
        size_t free_bytes = 0, all = 0;
        if (hipMemGetInfo(&free_bytes, &all) != hipSuccess || !decode_ahead_copy_fits(blocks, free_bytes)) { (void)hipGetLastError(); return FORGE_HIP_OK; }
    }
    // matrices of one depth, one behind the other, as PA_KQ blocks; false: no memory for them, and the other kernel takes the steps
    auto units = [&](const std::vector<const QWeight*>& ws, PaWeights* to) {
        size_t blocks = 0;
        for (const QWeight* w : ws) blocks += (size_t)w->N * (w->K / 32);
        uint8_t* codes = st->dev<uint8_t>(blocks * 32);
        uint32_t* words = codes ? st->dev<uint32_t>(blocks * 4) : nullptr;
        if (!words) { (void)hipGetLastError(); return false; }
        *to = PaWeights{codes, reinterpret_cast<const uint16_t*>(words)};
        for (const QWeight* w : ws) {
            pa_repack(*w, codes, words);
            codes += (size_t)w->N * w->K;
            words += (size_t)w->N * (w->K / 32);
        }
        return true;
    };
    for (size_t l = 0; l < layers.size(); l++) {
        const PdLayerIn& in = layers[l];
        if (kq) {
            const std::vector<const QWeight*> parts[4] = {{in.q, in.k, in.v}, {in.o}, {in.gate, in.up}, {in.down}};
            for (int k = 0; k < 4; k++)
                if (!units(parts[k], &host[l].w[k])) return FORGE_HIP_OK;
        } else {
            const QWeight* w[4] = {in.qkv, in.o, in.gate_up, in.down};
            for (int k = 0; k < 4; k++) host[l].w[k] = PaWeights{w[k]->qs, w[k]->scales};
        }
        host[l].norm[0] = in.attn_norm; host[l].norm[1] = in.ffn_norm; host[l].kc = in.kc; host[l].vc = in.vc;
    }
    host.back() = host[0];
    host.back().norm[0] = final_norm;
    PaLayer* dl = st->dev<PaLayer>(host.size() * sizeof(PaLayer));
    const size_t n_tagged = (size_t)H + QKS + 2 * KV + QKS / 32 * 9 + I / 32 * 9 + 2 * (size_t)st->grid + (size_t)c.heads * a.splits * (hd + 2);
    uint64_t* t = st->dev<uint64_t>(n_tagged * 8);
    if (!dl || !t) return fail(FORGE_HIP_ERR_HIP, "resident decode: out of device memory");
    FH_HIP(hipMemcpy(dl, host.data(), host.size() * sizeof(PaLayer), hipMemcpyHostToDevice));
    FH_HIP(hipMemset(t, 0, n_tagged * 8));                       // tag 0 is never expected
    st->tagged = t; st->tagged_bytes = n_tagged * 8;
    a.layers = dl;
    a.tx = t; t += H;
    a.tq = t; t += QKS;
    a.tkv = t; t += 2 * KV;
    a.taq = t; t += QKS / 32 * 9;
    a.taq2 = t; t += I / 32 * 9;
    a.tpart = t; t += 2 * (size_t)st->grid;
    a.trec = t;
    a.lm = PaWeights{lm_head.qs, lm_head.scales};
    if (kq) {
        if (!units({&lm_head}, &a.lm)) return FORGE_HIP_OK;
        FH_HIP(hipDeviceSynchronize());
        FH_HIP(hipGetLastError());
    }
    a.embed = embed; a.cos_t = cos_t; a.sin_t = sin_t;
    a.logits = logits; a.state = state; a.counts = counts; a.penalty = 1.0f;
    { const char* e = getenv("FORGE_HIP_PD_TAG_START"); if (e) a.tag_base = (uint32_t)strtoul(e, nullptr, 0); }
    pa_set_poll_limit(st.get(), 0);
    { const char* e = getenv("FORGE_HIP_PD_SPIN_LIMIT"); if (e && atoi(e) > 0) a.spin_limit = (uint32_t)atoi(e); }
    if (!(getenv("FORGE_HIP_PD_HOSTWORD") && getenv("FORGE_HIP_PD_HOSTWORD")[0] == '0')) {
        void *hp = nullptr, *dp = nullptr;
        if (hipHostMalloc(&hp, 64, hipHostMallocMapped) == hipSuccess) {
            if (hipHostGetDevicePointer(&dp, hp, 0) == hipSuccess) {
                st->host_out = static_cast<unsigned long long*>(hp);
                st->host_out_dev = static_cast<unsigned long long*>(dp);
                st->host_out[0] = 0;
            } else {
                (void)hipHostFree(hp);
            }
        }
        (void)hipGetLastError();
    }
    st->wall_khz = khz;
    st->n_stamps = 6 * a.L + 3;
    *out = st.release();
    return FORGE_HIP_OK;
}

void pa_set_poll_limit(PaState* st, uint32_t n) { st->args.spin_limit = n ? n : 400000u; }
void pa_set_kv_pages(PaState* st, const PageTable& pt, uint32_t max_seq) {
    st->args.pages = pt.table;
    st->args.page_shift = pt.shift;
    st->args.n_pages = pt.table ? max_seq >> pt.shift : 0u;
}
void pa_set_repeat_penalty(PaState* st, float penalty) { st->args.penalty = penalty; }

// Enqueues the step at position `pos` (which the device has in `state`) for `token`; `step_seq`: its number, not 0.  With `profile` the kernel also records the clock at the start of every phase.
int32_t pa_enqueue(PaState* st, int64_t pos, bool profile, uint32_t token, uint32_t step_seq, hipStream_t s) {
    PaArgs& a = st->args;
    a.token = token;
    a.step_seq = step_seq;
    a.host_out = st->host_out_dev;
    if (a.host_out) a.host_seq = ++st->seq;
    if (a.tag_base > 0xF0000000u) {      // tags are about to wrap: start again from zeroed buffers
        FH_HIP(hipMemsetAsync(st->tagged, 0, st->tagged_bytes, s));
        a.tag_base = 0;
    }
    if (profile && !a.stamps) {
        a.stamps = st->dev<unsigned long long>(st->n_stamps * 8);
        if (!a.stamps) return fail(FORGE_HIP_ERR_HIP, "resident decode: out of device memory");
    }
    unsigned long long* keep = a.stamps;
    if (!profile) a.stamps = nullptr;
    void* kargs[] = {&a};
    const hipError_t e = resident_launch(pos < (int64_t)st->one_rows ? st->kernel : st->kernel_long, st->grid, PA_THREADS, kargs, st->lds, st->cooperative, s);
    a.stamps = keep;
    if (e != hipSuccess) return fail(FORGE_HIP_ERR_HIP, std::string("resident decode launch: ") + hipGetErrorString(e));
    a.tag_base += 6 * a.L + 1;
    return FORGE_HIP_OK;
}

// The next token, from the word that the kernel writes last; false: not in use or not in time, wait for the stream instead.
bool pa_wait_token(PaState* st, uint32_t* next) {
    if (!st->host_out || !st->args.host_out) return false;
    const volatile unsigned long long* w = st->host_out;
    const auto t0 = std::chrono::steady_clock::now();
    for (uint32_t spin = 0;; spin++) {
        const unsigned long long v = *w;
        if ((uint32_t)(v >> 32) == st->seq) { *next = (uint32_t)v; return true; }
        if ((spin & 1023u) == 1023u && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(200)) return false;
    }
}

// After the stream has drained, with the abort flag: a step that gave up did not happen (the position advances last); what may have happened
// is the count of its token, which is taken back.
int32_t pa_after_sync(PaState* st, uint32_t abort_flag, hipStream_t s) {
    if (!abort_flag) return FORGE_HIP_OK;
    PaArgs& a = st->args;
    uint32_t seq = 0, n = 0;
    FH_HIP(hipMemcpyAsync(&seq, a.state + 4, 4, hipMemcpyDeviceToHost, s));
    FH_HIP(hipMemcpyAsync(&n, a.counts + a.token, 4, hipMemcpyDeviceToHost, s));
    FH_HIP(hipStreamSynchronize(s));
    if (seq == a.step_seq && n) {
        n -= 1;
        FH_HIP(hipMemcpyAsync(a.counts + a.token, &n, 4, hipMemcpyHostToDevice, s));
        FH_HIP(hipStreamSynchronize(s));
    }
    FH_HIP(hipMemsetAsync(st->tagged, 0, st->tagged_bytes, s));
    FH_HIP(hipMemsetAsync(a.state + 3, 0, 4, s));
    FH_HIP(hipStreamSynchronize(s));
    a.tag_base = 0;
    return fail(FORGE_HIP_ERR_HIP, "resident decode step gave up waiting for another workgroup's data (grid not co-resident?)");
}

// Milliseconds between the phase starts of the last profiled step, as pd_phase_ms reports them.
int32_t pa_phase_ms(PaState* st, std::vector<float>* out, hipStream_t s) {
    PaArgs& a = st->args;
    out->clear();
    if (!a.stamps) return FORGE_HIP_OK;
    st->stamps_host.resize(st->n_stamps);
    FH_HIP(hipMemcpyAsync(st->stamps_host.data(), a.stamps, st->n_stamps * 8, hipMemcpyDeviceToHost, s));
    FH_HIP(hipStreamSynchronize(s));
    for (uint32_t i = 0; i + 1 < st->n_stamps; i++)
        out->push_back((float)((double)(int64_t)(st->stamps_host[i + 1] - st->stamps_host[i]) / (double)st->wall_khz));
    return FORGE_HIP_OK;
}

}  // namespace fh
