// One decode token of a block network (block_model.hip) as ONE kernel: bfloat16 models, whose step is a chain of 90 to 210 products and attentions.  First small ones, that read almost
// nothing each; the wide form at the end is for layers that registers do not hold.
//
// As kernels in a graph a link of that chain is 2.4 to 6 us however small; here it is a hand-over of 1.2 us and what it computes (resident.h: tagged elements, bounded waits,
// a buffer is overwritten only by a phase whose inputs transitively depend on every reader of what it held).  The form is decode_ahead.hip's:
//   * The first G workgroups hold a layer's matrices in registers, in tiles of 16 rows: eight waves share out a tile's depth, four fetch vectors.  G is the fewest that
//     hold them (64 for both 135M shapes): a hand-over costs more among more workgroups.
//   * The matrices that follow the attention are requested while that is at work, and so are the next layer's.
//   * A head (latent attention, linear attention) or a key / value head (grouped attention) has a workgroup of its own, or several that share out its context, behind the G.  What
//     a head does between the input product and the output product has no hand-over but that of the parts: its small matrices (W_uq, W_uk, W_uv) are
//     in the registers of the workgroups that attend for it, and so are its cached rows, requested a layer ahead.
//   * All workgroups share the output matrix.
// A row times a vector is a product of 16 rows on the matrix unit.  Its other 15 columns are free, so a vector that the kernel sequence multiplies in 32-bit goes in as three
// bfloat16 planes (x = hi + lo + rest, exact) in columns of their own: the same precision, no conversion of weights and no reduction over lanes.
// An element past bfloat16's range would be no number in its planes, and what pads a product multiplies weights and cached rows by 0: both take numbers of ordinary size.  A model has them if
// no weight is larger than PB_LARGEST (2^32): a normed element is then below 2^40, a projection below 2^87, a gated head's output below 2^126.  A model with a larger weight, an infinity or a NaN
// keeps the sequence (limits on the elements themselves, two instructions each, cost 4 us of 406 a token).
//
// Per token in us, kernel sequence / this, by rows of context (sizes of vabirax_135m: 9 heads of 64 + 32, window 1024; kakirax_135m: three layers of linear attention to one of grouped):
//   latent            20: 886 / 389    200: 895 / 398    900: 900 / 421    2400: 901 / 422
//   linear, grouped   20: 647 / 402    200: 647 / 408    900: 648 / 412    2400: 648 / 421
// What bounds it: the chain.  A layer run of the first takes 13 us: input product 1.9, the heads 5.5 (0.6 of them the merge of eight parts), output product 1.5, gate;up 1.8, down 2.0, each
// of the products 0.4 to 1.2 of waiting for what was handed over, 0.4 on the matrix unit and 0.4 of sums, epilogue and store.  Its weights (7.7 MB) would take 1.6.  What
// decided the form, measured: branches around the pieces of a product (each read of the vector then waits for the one before) 502 -> 453 at 2400 rows; values transposed ahead of the query, and
// four waves a workgroup that attend, 453 -> 419; loop-invariant addresses kept over the layers (24 spilled registers) 532 -> 501.  Without effect: 96 to 160 workgroups
// for the matrices (415 to 419; linear 2 % faster with 128), the layer norm an element a thread of all twelve waves (414 -> 427: the matrices' waves poll behind their loads).
#include <stddef.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <memory>
#include <vector>

#include "common.h"
#include "decode_block.h"
#include "dense.h"
#include "device_utils.h"
#include "lds_transpose.h"
#include "resident.h"
#include "resident_seat.h"

namespace fh {

namespace {

constexpr uint32_t PB_POLL = 4, PB_COMP = 8, PB_WAVES = PB_POLL + PB_COMP, PB_THREADS = PB_WAVES * 64, PB_POLL_THREADS = PB_POLL * 64;
constexpr float PB_LOG2E = 1.4426950408889634f;
constexpr float PB_NO_KEYS = -3.0e38f;       // maximum of a part without keys: weight 0
// Limits of the narrow forms: tiles of 16 rows a workgroup, pieces of 32 columns a wave, and the heads' sizes below.  What they are bound by (one of them raised at a time, compiled, not measured):
// registers hold no longer cached row (PB_ROW 192 spills 16 bytes a lane) and LDS no longer latent (its transposed values are 120 KB of 159).  The others are the widths of the models at hand: one
// more tile or piece of a matrix (width 1024, feed-forward 2048) spills nothing in 143 to 161 registers of 168; nor do PB_QR 256 (a polling thread an element), PB_DIM 128 (dim and rot together: 16
// rows a wave, 192) and PB_VDIM 128.
constexpr int PB_TI = 2, PB_UI = 3;          // input product
constexpr int PB_UO = 3;                     // output product
constexpr int PB_TG = 3;                     // gate;up
constexpr int PB_UD = 6;                     // down
constexpr int PB_UL = 6;                     // the loop's input product
constexpr uint32_t PB_WIDTH = 32 * PB_COMP * PB_UI, PB_FF = 32 * PB_COMP * PB_UD;
constexpr int PB_HEAD_U = 6;                 // pieces of an output matrix's tile in each of two sets
// Attention: a wave takes PB_KEYS keys a round.
constexpr uint32_t PB_KEYS = 32, PB_SPLITS = 64;
constexpr uint32_t PB_CT = PB_KEYS + 8;      // LDS row of transposed values
// Latent heads: query latent, unrotated part, cached row, latent, values.
constexpr uint32_t PB_QR = 192, PB_DIM = 64, PB_ROW = 160, PB_RANK = 128, PB_VDIM = 64;
constexpr uint32_t PB_GROUP = 4;             // query heads of a key / value head
constexpr int PB_STATE = 3;                  // linear attention: pieces of 4 state elements a thread
constexpr uint32_t PB_LOW = 16, PB_LVDIM = 128;
constexpr uint32_t PB_LDS = 160 * 1024 - 1024;

enum PbKind : uint32_t { PB_FIRST, PB_GROUPED };      // PB_FIRST: latent or linear attention, whichever the design has

// T: tiles a workgroup; per: pieces of 32 columns a wave
struct PbMat { uint32_t N, K, tiles, T, per; };
struct PbLayer {
    const __bf16 *in, *o, *gate_up, *down;
    const float *norm1, *norm2, *post1, *post2, *next;   // weight, then bias `width` further on; post (elementwise norms only), next (what follows down, null: nothing)
    float alpha1, alpha2, post_alpha1, post_alpha2, next_alpha;
    uint32_t kind, loop;
    uint8_t *cache, *cache_v;                            // cache_v: grouped attention's values
    const __bf16 *uq, *uk, *uv;                          // latent attention; uk: transposed, [head][rank][dim]
    const float *wa, *wb, *wc;                           // latent: the norms of query and key / value latents; grouped: of q and k; linear: W2, its bias, the heads' norm
};

struct PbArgs {
    PbMat in[2], o[2], gate_up, down, loop, head;        // in, o: by PbKind
    uint32_t L, W, Wn, ff;
    uint32_t empty;                                      // where the words behind lie decides which scalars are loaded in one: without it 230 more reads of scalars kept in lanes, 420 -> 427 us a token (latent)
    uint32_t table_ld, table_n, G, act;
    uint32_t splits, splits_max, attend;                 // parts of a context; waves of a workgroup that attend
    LatentShape ls;
    GroupedShape gs;
    LinearShape ns;
    float eps, embed_scale, cap;
    const PbLayer* layers;
    const __bf16 *table, *head_w, *loop_w;
    const float* final_norm;
    const float *cos_t, *sin_t;
    // tagged exchange buffers
    uint64_t* th;      // elementwise norms: [W / 2] the next product's input, two bfloat16 to an element; layer norms: [W] the stream
    uint64_t* tl;      // [W / 2] likewise, behind the loop's input product
    uint64_t* traw;    // [input product's rows] in 32-bit, the activated gates among them
    uint64_t* trec;    // [heads][splits][(values + 2) per query head] weighted sum, maximum and weight sum of a part
    uint64_t* tout;    // the heads' output: two bfloat16 to an element; linear attention: 32-bit
    uint64_t* tact;    // [ff / 2] act(gate) * up, two bfloat16 to an element
    uint64_t* tpart;   // [2 workgroups of the grid]  argmax candidates
    float* logits;
    uint32_t* state;   // [0] position  [1] token  [2] next token  [3] abort flag  [4] number of the step that counted its token
    uint32_t* counts;
    float penalty;
    uint32_t tag_base, spin_limit, token, step_seq;
    unsigned long long* host_out;
    uint32_t host_seq;
    unsigned long long* stamps;
    uint32_t plane, off_red, off_stats, off_layers, off_attn, off_in;      // plane: elements of a vector's plane (bytes 0 .. 4 planes); LDS byte offsets
};
// Tags of a layer run, behind its base.
enum PbTag : uint32_t { PB_T_LOOP = 1, PB_T_RAW, PB_T_REC, PB_T_OUT, PB_T_O, PB_T_ACT, PB_T_DOWN, PB_TAGS };

__device__ __forceinline__ uint32_t pb_sgpr(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }
// Pointers of a layer, from their copy in LDS.
template <typename T>
__device__ __forceinline__ T* pb_ptr(T* const& p) {
    const uint64_t v = *reinterpret_cast<const uint64_t*>(&p);
    return reinterpret_cast<T*>(((uint64_t)pb_sgpr((uint32_t)(v >> 32)) << 32) | pb_sgpr((uint32_t)v));
}
__device__ __forceinline__ v8bf pb_load8(const __bf16* base, uint32_t off) {
    return __builtin_bit_cast(v8bf, ldg(reinterpret_cast<const uint4*>(reinterpret_cast<const uint8_t*>(base) + off)));
}
__device__ __forceinline__ float pb_f32(const float* base, uint32_t i) { return ldg(base + i); }

// Three bfloat16 that add up to x.
__device__ __forceinline__ void pb_split(float x, __bf16& hi, __bf16& lo, __bf16& rest) {
    hi = (__bf16)x;
    const float r = x - (float)hi;
    lo = (__bf16)r;
    rest = (__bf16)(r - (float)lo);
}
__device__ __forceinline__ uint32_t pb_pack(float a, float b) {
    return (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)a) | (uint32_t)__builtin_bit_cast(uint16_t, (__bf16)b) << 16;
}
// Columns 0 .. 3 of a product (the planes of its vector, the last one zero) as their sum, in all of them.
__device__ __forceinline__ v4f pb_columns(v4f v) {
#pragma unroll
    for (int r = 0; r < 4; r++) v[r] = lane_xor_add<2>(lane_xor_add<1>(v[r]));
    return v;
}

// A wave's part of a matrix: pieces c * per .. of T tiles.  What lies past the matrix re-reads its last piece or row: no condition around a load.
__device__ __forceinline__ PbMat pb_of(const PbMat (&m)[2], uint32_t kind) { return kind == PB_FIRST ? m[0] : m[1]; }
template <int T, int U> struct PbSet { v8bf f[T][U]; };
template <int T, int U>
__device__ __forceinline__ void pb_load(PbSet<T, U>& s, const __bf16* w, const PbMat& m, uint32_t wg, uint32_t c, uint32_t lane) {
    asm volatile("" : "+v"(lane));           // the addresses are worked out here: kept from layer to layer they would not fit the registers
    const uint32_t last = m.K / 32 - 1;
#pragma unroll
    for (int t = 0; t < T; t++) {
        const uint32_t tile = min(wg * m.T + min((uint32_t)t, m.T - 1), m.tiles - 1);
        const uint32_t at = min(tile * 16 + (lane & 15u), m.N - 1) * m.K * 2 + (lane >> 4) * 16;
#pragma unroll
        for (int i = 0; i < U; i++) s.f[t][i] = pb_load8(w, at + min(c * m.per + min((uint32_t)i, m.per - 1), last) * 64);
    }
}
// x: this lane's column of the vector, from element 8 (lane / 16) on; zeros: as many zeros.  Pieces that are not the wave's meet zeros: with no branch between them all
// reads of the vector are on their way before the first product.
template <int T, int U>
__device__ __forceinline__ void pb_mul(const PbSet<T, U>& s, const PbMat& m, uint32_t c, const __bf16* x, const __bf16* zeros, v4f (&acc)[T]) {
    v8bf b[U];
#pragma unroll
    for (int i = 0; i < U; i++) {
        const uint32_t k = c * m.per + i;
        b[i] = load8((uint32_t)i < m.per && k < m.K / 32 ? x + 32 * k : zeros);
    }
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < U; i++)
#pragma unroll
        for (int t = 0; t < T; t++) acc[t] = mma16(s.f[t][i], b[i], acc[t]);
}

// Vectors, fetched by the polling waves: bfloat16 pairs into the first plane, or 32-bit elements into three; zeros behind them up to `total`.
template <int N>
__device__ __forceinline__ void pb_fetch_pairs(const uint64_t* t, uint32_t tag, uint32_t n, uint32_t total, uint32_t* plane, const PollCtx& cx) {
    uint32_t v[N];
    poll_tagged<N>([&](int i) { return t + min(cx.tid + i * PB_POLL_THREADS, n - 1); }, [&](int) { return tag; }, v, cx);
#pragma unroll
    for (int i = 0; i < N; i++) {
        const uint32_t e = cx.tid + i * PB_POLL_THREADS;
        if (e < total) plane[e] = e < n ? v[i] : 0u;
    }
}
__device__ __forceinline__ void pb_put(__bf16* x, uint32_t plane, uint32_t e, float v) {
    pb_split(v, x[e], x[plane + e], x[2 * plane + e]);
}
template <int N>
__device__ __forceinline__ void pb_fetch_floats(const uint64_t* t, uint32_t tag, uint32_t n, uint32_t total, __bf16* x, uint32_t plane, const PollCtx& cx) {
    uint32_t v[N];
    poll_tagged<N>([&](int i) { return t + min(cx.tid + i * PB_POLL_THREADS, n - 1); }, [&](int) { return tag; }, v, cx);
#pragma unroll
    for (int i = 0; i < N; i++) {
        const uint32_t e = cx.tid + i * PB_POLL_THREADS;
        if (e < total) pb_put(x, plane, e, e < n ? __uint_as_float(v[i]) : 0.f);
    }
}
__device__ __forceinline__ float pb_tanh(float alpha, float x, float w, float b) { return tanhf(alpha * x) * w + b; }
__device__ __forceinline__ float pb_embed(const PbArgs& a, uint32_t e) {
    const float v = (float)__builtin_bit_cast(__bf16, ldg(reinterpret_cast<const uint16_t*>(a.table) + (size_t)a.token * a.table_ld + min(e, a.table_n - 1))) * a.embed_scale;
    return e < a.table_n ? v : 0.f;
}

// ---- attention over cached rows --------------------------------------------------------------------------------------------------
// The rows of a wave's keys: two tiles of 16 keys, CK pieces of 32 columns; VK pieces of a value row (latent attention: the key's first ones).
template <int CK, int VK, bool LATENT>
struct PbKeys {
    v8bf k[2][CK], v[LATENT ? 1 : 2][LATENT ? 1 : VK];
    // keys first .. first + 31, those from `pos` on as the last cached one
    __device__ __forceinline__ void load(const uint8_t* kb, uint32_t k_bytes, const uint8_t* vb, uint32_t v_bytes, uint32_t nk, uint32_t nv, uint32_t first, uint32_t pos, uint32_t lane) {
        asm volatile("" : "+v"(lane));
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const uint32_t row = min(first + 16 * t + (lane & 15u), pos - 1), at = (lane >> 4) * 16;
#pragma unroll
            for (int s = 0; s < CK; s++) k[t][s] = pb_load8((const __bf16*)kb, row * k_bytes + at + min((uint32_t)s, nk - 1) * 64);
            if constexpr (!LATENT) {
#pragma unroll
                for (int s = 0; s < VK; s++) v[t][s] = pb_load8((const __bf16*)vb, row * v_bytes + at + min((uint32_t)s, nv - 1) * 64);
            }
        }
    }
    __device__ __forceinline__ const v8bf& value(int t, int s) const { if constexpr (LATENT) return k[t][s]; else return v[t][s]; }
    // The values, transposed, into the wave's own LDS: ahead of the query, which it has nothing to do with.
    __device__ __forceinline__ void lay_down(__bf16* ct, uint32_t lane) const {
#pragma unroll
        for (int t = 0; t < 2; t++)
#pragma unroll
            for (int i = 0; i < VK; i++) lay_down_transposed<__bf16, PB_CT>(ct, value(t, i), 32 * i, 16 * t, lane & 15u, lane >> 4);
    }
};
// A wave's running maximum (base 2), weight sum and weighted values; a lane: query head lane % 16.
template <int VK> struct PbRun { float m, l; v4f o[2 * VK]; };

// Keys first .. first + 31 of positions up to pos, whose own row is in LDS (fresh_k, fresh_v); the cached rows' values are in ct.  q: this lane's query head, from element 8 (lane / 16) on; ct, p: the wave's own LDS;
// p_row: a lane's row of it (one head: everybody's the same).  q is zero
// past the row's pieces; what there is past a row's own in the registers meets those zeros, or is not looked at (no branches: the reads of LDS would wait for each other).
template <int CK, int VK, bool LATENT>
__device__ __forceinline__ void pb_attend(PbKeys<CK, VK, LATENT>& kv, PbRun<VK>& run, uint32_t first, uint32_t pos, uint32_t nk, const __bf16* q, const __bf16* fresh_k,
                                          const __bf16* fresh_v, __bf16* ct, __bf16* p, uint32_t p_row, float c2, uint32_t lane) {
    const uint32_t l16 = lane & 15u, lg = lane >> 4;
    v4f s[2];
    float mx = -INFINITY;
    v8bf qf[CK];
#pragma unroll
    for (int i = 0; i < CK; i++) qf[i] = load8(q + 32 * i);
#pragma unroll
    for (int t = 0; t < 2; t++) {
        const uint32_t key = first + 16 * t + l16;
        if (first + 16 * t <= pos && pos < first + 16 * t + 16) {
#pragma unroll
            for (int i = 0; i < CK; i++) {
                const v8bf f = load8(fresh_k + 32 * min((uint32_t)i, nk - 1) + 8 * lg);
                if (key == pos) kv.k[t][i] = f;
            }
            for (uint32_t d = lane; d < 32 * VK; d += 64) ct[d * PB_CT + (pos - first)] = fresh_v[d];
        }
        s[t] = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < CK; i++) s[t] = mma16(kv.k[t][i], qf[i], s[t]);
        // register r: key first + 16 t + 4 lg + r
#pragma unroll
        for (int r = 0; r < 4; r++) {
            s[t][r] = first + 16 * t + 4 * lg + r <= pos ? s[t][r] * c2 : -INFINITY;
            mx = fmaxf(mx, s[t][r]);
        }
    }
    mx = lane_xor_max<32>(lane_xor_max<16>(mx));                     // finite: the first key is visible
    const float m_new = fmaxf(run.m, mx), alpha = __builtin_amdgcn_exp2f(run.m - m_new);
    run.m = m_new;
    run.l *= alpha;
#pragma unroll
    for (int t = 0; t < 2; t++) {
        float e[4];
#pragma unroll
        for (int r = 0; r < 4; r++) { e[r] = __builtin_amdgcn_exp2f(s[t][r] - m_new); run.l += e[r]; }
        if (!LATENT || l16 == 0) store4<__bf16>(p + p_row * PB_CT + 16 * t + 4 * lg, e[0], e[1], e[2], e[3]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");           // LDS operations of one wave execute in order
    __builtin_amdgcn_wave_barrier();
    const v8bf w = load8(p + p_row * PB_CT + 8 * lg);
#pragma unroll
    for (int i = 0; i < 2 * VK; i++) {
        run.o[i] *= alpha;
        run.o[i] = mma16(load8(ct + (16 * i + l16) * PB_CT + 8 * lg), w, run.o[i]);
    }
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// LDS of a workgroup that attends, VD values for each of H heads.
template <uint32_t VD, uint32_t H, uint32_t WAVES>
struct PbMerge {
    float o[WAVES][H][VD], m[WAVES][H], l[WAVES][H];
};
struct PbLatentLds {
    alignas(16) __bf16 ct[PB_WAVES][PB_RANK * PB_CT];
    alignas(16) __bf16 p[PB_WAVES][PB_CT];
    // zero past what a shape fills
    alignas(16) __bf16 x[4][PB_QR];          // planes: the normed query latent, then the merged latents
    alignas(16) __bf16 q[PB_DIM], row[PB_ROW], fresh[PB_ROW];      // unrotated query; the query against a cached row; this position's row
    float raw[PB_QR + PB_ROW + PB_VDIM];
    float out[PB_VDIM];
    PbMerge<PB_RANK, 1, PB_WAVES> merge;
};
template <uint32_t WAVES>
struct PbGroupedLds {
    alignas(16) __bf16 ct[WAVES][64 * PB_CT];
    alignas(16) __bf16 p[WAVES][16 * PB_CT];
    alignas(16) __bf16 q[16][64 + 8];
    alignas(16) __bf16 k[64], v[64];
    float raw[(PB_GROUP + 2) * 64 + PB_GROUP * 64];
    PbMerge<64, PB_GROUP, WAVES> merge;
};
template <uint32_t WAVES>
struct PbLinearLds {
    float raw[2 * 64 + 2 * PB_LVDIM + PB_LOW];
    float a[64];
    alignas(16) v4f part[WAVES][PB_LVDIM / 4];
};
template <uint32_t WAVES>
struct PbKakiraxLds {
    PbGroupedLds<WAVES> grouped;
    PbLinearLds<WAVES> linear;
};

// The waves' sums as the workgroup's part, thread t: head t / VD, value t % VD.  w: the part's weight sum.
struct PbPart { float o, m, l; };
template <uint32_t VD, uint32_t H, uint32_t WAVES>
__device__ __forceinline__ PbPart pb_waves(const PbMerge<VD, H, WAVES>& sh, uint32_t waves, uint32_t head, uint32_t d) {
    PbPart p{0.f, PB_NO_KEYS, 0.f};
#pragma unroll 4
    for (uint32_t w = 0; w < waves; w++) p.m = fmaxf(p.m, sh.m[w][head]);
#pragma unroll 4
    for (uint32_t w = 0; w < waves; w++) {
        const float e = __builtin_amdgcn_exp2f(sh.m[w][head] - p.m);
        p.o = fmaf(e, sh.o[w][head][d], p.o);
        p.l = fmaf(e, sh.l[w][head], p.l);
    }
    return p;
}
template <int VK, uint32_t VD, uint32_t H, uint32_t WAVES>
__device__ __forceinline__ void pb_leave(PbMerge<VD, H, WAVES>& sh, const PbRun<VK>& run, uint32_t heads, uint32_t wave, uint32_t lane) {
    const uint32_t l16 = lane & 15u, lg = lane >> 4;
    const float l = lane_xor_add<32>(lane_xor_add<16>(run.l));
    if (l16 >= heads) return;
#pragma unroll
    for (int i = 0; i < 2 * VK; i++)
        *reinterpret_cast<v4f*>(&sh.o[wave][l16][16 * i + 4 * lg]) = run.o[i];
    if (lg == 0) {
        sh.m[wave][l16] = run.m;
        sh.l[wave][l16] = l;
    }
}

// The parts of `heads` heads: everybody but the first hands its part over, the first adds all up.  Thread t < heads * vd: head t / vd, value t % vd; returns its
// weighted mean (first only).  False: the step is given up.
template <uint32_t VD, uint32_t H, uint32_t WAVES>
__device__ __forceinline__ bool pb_parts(const PbArgs& a, const PbMerge<VD, H, WAVES>& sh, uint32_t owner, uint32_t split, uint32_t heads, uint32_t vd, uint32_t tag, float* recs, float& mean,
                                         const PollCtx& cx) {
    const uint32_t n = heads * vd, rec = heads * (vd + 2), head = cx.tid / vd, d = cx.tid - head * vd;
    PbPart p{0.f, PB_NO_KEYS, 1.f};
    if (cx.tid < n) p = pb_waves(sh, a.attend, head, d);
    uint64_t* out = a.trec + (size_t)owner * a.splits_max * rec;
    if (split > 0) {
        uint64_t* mine = out + (size_t)split * rec + head * (vd + 2);
        if (cx.tid < n) {
            stc64(mine + d, tag, __float_as_uint(p.o));
            if (d < 2) stc64(mine + vd + d, tag, __float_as_uint(d == 0 ? p.m : p.l));
        }
        return true;
    }
    if (a.splits > 1) {
        const uint32_t ne = (a.splits - 1) * rec;
        constexpr int N = 4;
        if (cx.wave < PB_POLL) {
            for (uint32_t e0 = 0; e0 < ne; e0 += N * PB_POLL_THREADS) {
                uint32_t v[N];
                poll_tagged<N>([&](int i) { return out + rec + min(e0 + cx.tid + i * PB_POLL_THREADS, ne - 1); }, [&](int) { return tag; }, v, cx);
#pragma unroll
                for (int i = 0; i < N; i++)
                    if (e0 + cx.tid + i * PB_POLL_THREADS < ne) recs[e0 + cx.tid + i * PB_POLL_THREADS] = __uint_as_float(v[i]);
            }
        }
        __syncthreads();
        if (*cx.sh_abort) return false;
        if (cx.tid < n) {
            // eight parts at a time, all of them read before the first is used; behind the last one it again, with weight 0
            const float* r = recs + head * (vd + 2);
            const uint32_t others = a.splits - 1;
            constexpr uint32_t B = 8;
            float o = p.o, l = p.l, m = p.m;
            for (uint32_t s0 = 0; s0 < others; s0 += B) {
                float ms[B], os[B], sums[B], m_new = m;
#pragma unroll
                for (uint32_t i = 0; i < B; i++) {
                    const float* q = r + min(s0 + i, others - 1) * rec;
                    ms[i] = q[vd]; sums[i] = q[vd + 1]; os[i] = q[d];
                }
#pragma unroll
                for (uint32_t i = 0; i < B; i++) m_new = fmaxf(m_new, ms[i]);
                const float e = __builtin_amdgcn_exp2f(m - m_new);
                m = m_new;
                o *= e;
                l *= e;
#pragma unroll
                for (uint32_t i = 0; i < B; i++) {
                    const float w = s0 + i < others ? __builtin_amdgcn_exp2f(ms[i] - m) : 0.f;
                    o = fmaf(w, os[i], o);
                    l = fmaf(w, sums[i], l);
                }
            }
            p.o = o;
            p.l = l;
        }
        // recs lies where a wave that is done lays down the next layer's values (one head: a barrier of its caller's comes before that).  Here rather than behind the store of the result, where
        // fewer waves wait for it: 399 us a token against 401 (kakirax_135m, 20 rows, where nothing is merged: the code around it comes out better).
        if constexpr (H > 1) __syncthreads();
    }
    mean = p.o / p.l;
    return true;
}

// The first key that position pos sees, and a workgroup's first key of a round.
__device__ __forceinline__ uint32_t pb_lo(uint32_t window, uint32_t pos) { return window && pos >= window ? pos - window + 1 : 0u; }

// ---- latent attention: a workgroup per (head, part) --------------------------------------------------------------------------------
// [norms, cache row | W_uq, rotation | W_uk^T | attention | merge | W_uv * gate]
__device__ __forceinline__ bool pb_latent_layers(const PbArgs& a, const PbLayer* layers, PbLatentLds* sh, float* recs, uint32_t pos, PollCtx& cx) {
    const LatentShape& s = a.ls;
    const uint32_t role = cx.wg - a.G, head = role / a.splits, split = role - head * a.splits;
    const uint32_t wave = cx.wave;
    const uint32_t nq = s.q_rank / 32, nd = s.dim / 32, nk = s.cache_row() / 32, nv = s.rank / 32, rows = s.dim + s.rot;
    const uint32_t lo = pb_lo(s.window, pos), span = PB_KEYS * a.attend, first0 = wave < a.attend ? lo + split * span + wave * PB_KEYS : 0xFFFFFFFFu,
                   step = a.splits * span;
    const float c2 = s.scale * PB_LOG2E;
    // the rotation of the query's rows 16 wave + 4 lg + .., and of this thread's element of the cache row
    float qc[2], qs[2], fc = 1.f, fs = 0.f;
    {
        const uint32_t lg = cx.lane >> 4, fi = cx.tid - PB_POLL_THREADS;
        const float *ct = a.cos_t + (size_t)pos * s.rot_pairs, *st = a.sin_t + (size_t)pos * s.rot_pairs;
#pragma unroll
        for (uint32_t i = 0; i < 2; i++) {
            const uint32_t j = 16 * wave + 4 * lg + 2 * i, pair = (j - s.dim) / 2;
            const bool turns = j >= s.dim && j < rows && pair < s.rot_pairs;
            qc[i] = turns ? ldg(ct + pair) : 1.f;
            qs[i] = turns ? ldg(st + pair) : 0.f;
        }
        const uint32_t pair = (fi - s.rank) / 2;
        if (fi >= s.rank && fi < s.cache_row() && pair < s.rot_pairs) { fc = ldg(ct + pair); fs = ldg(st + pair); }
    }
#pragma nounroll
    for (uint32_t l = 0; l < a.L; l++) {
        // The thread's number is read afresh in every layer: addresses that follow from it would be kept from layer to layer and not fit the registers.
        asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
        const PbLayer& L = layers[l];
        const uint32_t base = a.tag_base + l * PB_TAGS, lane = cx.lane, tid = cx.tid, l16 = lane & 15u, lg = lane >> 4;
        const uint32_t fi = tid - PB_POLL_THREADS;                   // element of the cache row: threads of the fifth wave on
        // requested as soon as the layer before is done: the cached rows and the head's matrices
        PbKeys<PB_ROW / 32, PB_RANK / 32, true> kv;
        if (first0 <= pos) kv.load(pb_ptr(L.cache), s.cache_row() * 2, nullptr, 0, nk, nv, first0, pos, lane);
        v8bf uq[PB_QR / 32], uk[PB_DIM / 32];
        {
            const uint32_t r = min(16 * wave + l16, rows - 1);
            const __bf16* w = pb_ptr(L.uq);
#pragma unroll
            for (uint32_t i = 0; i < PB_QR / 32; i++) uq[i] = pb_load8(w, ((head * rows + r) * s.q_rank + 32 * min(i, nq - 1) + 8 * lg) * 2);
            const uint32_t rr = min(16 * wave + l16, s.rank - 1);
            w = pb_ptr(L.uk);
#pragma unroll
            for (uint32_t i = 0; i < PB_DIM / 32; i++) uk[i] = pb_load8(w, ((head * s.rank + rr) * s.dim + 32 * min(i, nd - 1) + 8 * lg) * 2);
        }
        const float nw = wave < PB_POLL ? pb_f32(pb_ptr(L.wa), min(tid, s.q_rank - 1)) : pb_f32(pb_ptr(L.wb), min(fi, s.rank - 1));
        if (first0 <= pos) kv.lay_down(sh->ct[wave], lane);
        // ---- the raw projections
        if (wave < PB_POLL) {
            const uint32_t n = s.raw_row(), ne = n + s.vdim;
            constexpr int N = 2;
            static_assert(PB_QR + PB_ROW + PB_VDIM <= N * PB_POLL_THREADS, "fetched at once");
            uint32_t v[N];
            auto at = [&](uint32_t e) { return a.traw + (e < n ? e : n + head * s.vdim + (e - n)); };
            poll_tagged<N>([&](int i) { return at(min(cx.tid + i * PB_POLL_THREADS, ne - 1)); }, [&](int) { return base + PB_T_RAW; }, v, cx);
#pragma unroll
            for (int i = 0; i < N; i++)
                if (cx.tid + i * PB_POLL_THREADS < ne) sh->raw[cx.tid + i * PB_POLL_THREADS] = __uint_as_float(v[i]);
        }
        __syncthreads();
        if (*cx.sh_abort) return false;
        // ---- norms: every wave sums for itself
        if (wave < PB_POLL) {
            float ss = 0.f;
#pragma unroll
            for (uint32_t i = 0; i < PB_QR; i += 64) {
                const float v = sh->raw[lane + i];
                if (lane + i < s.q_rank) ss = fmaf(v, v, ss);
            }
            const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)s.q_rank_n + s.eps);
            if (tid < PB_QR) pb_put(&sh->x[0][0], PB_QR, tid, tid < s.q_rank ? sh->raw[tid] * inv * nw : 0.f);
        } else if (fi < PB_POLL_THREADS) {
            const float* c = sh->raw + s.q_rank;
            float ss = 0.f;
#pragma unroll
            for (uint32_t i = 0; i < PB_RANK; i += 64) {
                const float v = c[lane + i];
                if (lane + i < s.rank) ss = fmaf(v, v, ss);
            }
            const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)s.rank_n + s.eps);
            if (fi < s.cache_row()) {
                float v;
                if (fi < s.rank) v = c[fi] * inv * nw;
                else v = fi & 1u ? c[fi] * fc + c[fi - 1] * fs : c[fi] * fc - c[fi + 1] * fs;
                const __bf16 b = (__bf16)v;
                sh->fresh[fi] = b;
                if (head == 0 && split == 0) stg(reinterpret_cast<uint16_t*>(pb_ptr(L.cache)) + (size_t)pos * s.cache_row() + fi, __builtin_bit_cast(uint16_t, b));
            }
        }
        __syncthreads();
        // ---- the query
        if (16 * wave < rows) {
            v4f acc = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t i = 0; i < PB_QR / 32; i++) acc = mma16(uq[i], load8(&sh->x[l16 & 3u][32 * i + 8 * lg]), acc);
            acc = pb_columns(acc);
            const uint32_t j = 16 * wave + 4 * lg;
            const float q0 = acc[0] * qc[0] - acc[1] * qs[0], q1 = acc[1] * qc[0] + acc[0] * qs[0], q2 = acc[2] * qc[1] - acc[3] * qs[1], q3 = acc[3] * qc[1] + acc[2] * qs[1];
            if (l16 == 0) store4<__bf16>(j < s.dim ? sh->q + j : sh->row + s.rank + (j - s.dim), q0, q1, q2, q3);
        }
        __syncthreads();
        if (16 * wave < s.rank) {
            v4f acc = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t i = 0; i < PB_DIM / 32; i++) acc = mma16(uk[i], load8(sh->q + 32 * i + 8 * lg), acc);
            if (l16 == 0) store4<__bf16>(sh->row + 16 * wave + 4 * lg, acc[0], acc[1], acc[2], acc[3]);
        }
        __syncthreads();
        // W_uv takes the place of W_uq while the heads attend
        v8bf uv[PB_RANK / 32];
        {
            const __bf16* w = pb_ptr(L.uv);
            const uint32_t r = min(16 * wave + l16, s.vdim - 1);
#pragma unroll
            for (uint32_t i = 0; i < PB_RANK / 32; i++) uv[i] = pb_load8(w, ((head * s.vdim + r) * s.rank + 32 * min(i, nv - 1) + 8 * lg) * 2);
        }
        // ---- attention
        PbRun<PB_RANK / 32> run;
        run.m = PB_NO_KEYS;
        run.l = 0.f;
#pragma unroll
        for (uint32_t i = 0; i < PB_RANK / 16; i++) run.o[i] = (v4f){0.f, 0.f, 0.f, 0.f};
        // (The first round outside the loop: inside, its rows would be waited for together with all that was requested behind them.)
        auto attend = [&](uint32_t first) { pb_attend(kv, run, first, pos, nk, sh->row + 8 * lg, sh->fresh, sh->fresh, sh->ct[wave], sh->p[wave], 0u, c2, lane); };
        if (first0 <= pos) attend(first0);
#pragma nounroll
        for (uint32_t first = first0; first <= pos && (first += step) <= pos;) {
            kv.load(pb_ptr(L.cache), s.cache_row() * 2, nullptr, 0, nk, nv, first, pos, lane);
            kv.lay_down(sh->ct[wave], lane);
            attend(first);
        }
        if (wave < a.attend) pb_leave(sh->merge, run, 1u, wave, lane);
        __syncthreads();
        float mean = 0.f;
        if (!pb_parts(a, sh->merge, head, split, 1u, s.rank, base + PB_T_REC, recs, mean, cx)) return false;
        if (split > 0) continue;
        // ---- values
        if (tid < PB_RANK) pb_put(&sh->x[0][0], PB_QR, tid, tid < s.rank ? mean : 0.f);
        __syncthreads();
        if (16 * wave < s.vdim) {
            v4f acc = (v4f){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (uint32_t i = 0; i < PB_RANK / 32; i++) acc = mma16(uv[i], load8(&sh->x[l16 & 3u][32 * i + 8 * lg]), acc);
            acc = pb_columns(acc);
            if (l16 == 0) *reinterpret_cast<v4f*>(sh->out + 16 * wave + 4 * lg) = acc;
        }
        __syncthreads();
        if (tid < s.vdim / 2) {
            const float* g = sh->raw + s.raw_row() + 2 * tid;
            stc64(a.tout + head * (s.vdim / 2) + tid, base + PB_T_OUT, pb_pack(sh->out[2 * tid] * g[0], sh->out[2 * tid + 1] * g[1]));
        }
        if (a.stamps && role == 0 && tid == 0) a.stamps[5 * l + 2] = wall_clock64();
    }
    return true;
}

// ---- grouped attention: a workgroup per (key / value head, part) -------------------------------------------------------------------
// [norms, rotation, cache row | attention | merge * gate]
template <uint32_t WAVES>
__device__ __forceinline__ bool pb_grouped_layer(const PbArgs& a, const PbLayer& L, PbGroupedLds<WAVES>* sh, float* recs, uint32_t role, uint32_t l, uint32_t pos, PollCtx& cx) {
    const GroupedShape& s = a.gs;
    const uint32_t kvh = role / a.splits, split = role - kvh * a.splits, group = s.group();
    const uint32_t lane = cx.lane, l16 = lane & 15u, lg = lane >> 4, wave = cx.wave, tid = cx.tid, base = a.tag_base + l * PB_TAGS;
    const uint32_t nk = s.dim / 32, nv = s.vdim / 32, span = PB_KEYS * a.attend, first0 = wave < a.attend ? split * span + wave * PB_KEYS : 0xFFFFFFFFu, step = a.splits * span;
    uint8_t *kc = pb_ptr(L.cache), *vc = pb_ptr(L.cache_v);
    PbKeys<2, 2, false> kv;
    auto load = [&](uint32_t first) { kv.load(kc + kvh * s.dim * 2, s.k_row() * 2, vc + kvh * s.vdim * 2, s.v_row() * 2, nk, nv, first, pos, lane); };
    if (first0 <= pos) load(first0);
    // norms and rotation: 16 lanes to a head, four elements a lane; the heads of the group, then the key
    const uint32_t nh = tid >> 4, sub = tid & 15u;
    float nw[4], rc[2], rs[2];
    {
        const float* w = nh < group ? pb_ptr(L.wa) : pb_ptr(L.wb);
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) nw[i] = pb_f32(w, min(4 * sub + i, s.dim - 1));
#pragma unroll
        for (uint32_t i = 0; i < 2; i++) {
            const uint32_t pair = min(2 * sub + i, s.rot_pairs - 1);
            const float c = ldg(a.cos_t + (size_t)pos * s.rot_pairs + pair), t = ldg(a.sin_t + (size_t)pos * s.rot_pairs + pair);
            rc[i] = 2 * sub + i < s.rot_pairs ? c : 1.f;
            rs[i] = 2 * sub + i < s.rot_pairs ? t : 0.f;
        }
    }
    if (first0 <= pos) kv.lay_down(sh->ct[wave], lane);
    const uint32_t gd = group * s.dim, ge = gd + s.dim, gv = ge + s.vdim, ne = gv + group * s.vdim;
    if (wave < PB_POLL) {
        constexpr int N = 3;
        static_assert((2 * PB_GROUP + 2) * 64 <= N * PB_POLL_THREADS, "fetched at once");
        uint32_t v[N];
        auto at = [&](uint32_t e) {
            const uint32_t k0 = s.heads * s.dim, v0 = k0 + s.k_row(), g0 = s.raw_row();
            return a.traw + (e < gd ? kvh * gd + e : e < ge ? k0 + kvh * s.dim + (e - gd) : e < gv ? v0 + kvh * s.vdim + (e - ge) : g0 + kvh * group * s.vdim + (e - gv));
        };
        poll_tagged<N>([&](int i) { return at(min(cx.tid + i * PB_POLL_THREADS, ne - 1)); }, [&](int) { return base + PB_T_RAW; }, v, cx);
#pragma unroll
        for (int i = 0; i < N; i++)
            if (cx.tid + i * PB_POLL_THREADS < ne) sh->raw[cx.tid + i * PB_POLL_THREADS] = __uint_as_float(v[i]);
    }
    __syncthreads();
    if (*cx.sh_abort) return false;
    if (nh <= group) {
        const bool in = 4 * sub < s.dim;
        v4f x = (v4f){0.f, 0.f, 0.f, 0.f};
        if (in) {
#pragma unroll
            for (uint32_t i = 0; i < 4; i++) x[i] = sh->raw[nh * s.dim + 4 * sub + i];      // zero past dim_n
        }
        float ss = (x[0] * x[0] + x[1] * x[1]) + (x[2] * x[2] + x[3] * x[3]);
        ss = lane_xor_add<1>(lane_xor_add<2>(lane_xor_add<4>(lane_xor_add<8>(ss))));
        const float inv = 1.0f / sqrtf(ss / (float)s.dim_n + s.eps);
#pragma unroll
        for (int i = 0; i < 4; i++) x[i] = x[i] * inv * nw[i];
        if (in) {
            const float y[4] = {x[0] * rc[0] - x[1] * rs[0], x[1] * rc[0] + x[0] * rs[0], x[2] * rc[1] - x[3] * rs[1], x[3] * rc[1] + x[2] * rs[1]};
            store4<__bf16>((nh < group ? sh->q[nh] : sh->k) + 4 * sub, y[0], y[1], y[2], y[3]);
            if (nh == group && split == 0) {
                const uint2 b = make_uint2(pb_pack(y[0], y[1]), pb_pack(y[2], y[3]));
                stg(reinterpret_cast<uint64_t*>(kc + ((size_t)pos * s.k_row() + kvh * s.dim) * 2) + sub, ((uint64_t)b.y << 32) | b.x);
            }
        }
    } else if (wave == (WAVES > PB_POLL ? PB_POLL : WAVES - 1)) {
        for (uint32_t i = lane; i < s.vdim; i += 64) {
            const __bf16 b = (__bf16)sh->raw[ge + i];
            sh->v[i] = b;
            if (split == 0) stg(reinterpret_cast<uint16_t*>(vc) + (size_t)pos * s.v_row() + kvh * s.vdim + i, __builtin_bit_cast(uint16_t, b));
        }
    }
    __syncthreads();
    PbRun<2> run;
    run.m = PB_NO_KEYS;
    run.l = 0.f;
#pragma unroll
    for (int i = 0; i < 4; i++) run.o[i] = (v4f){0.f, 0.f, 0.f, 0.f};
    auto attend = [&](uint32_t first) { pb_attend(kv, run, first, pos, nk, &sh->q[l16][8 * lg], sh->k, sh->v, sh->ct[wave], sh->p[wave], l16, s.scale * PB_LOG2E, lane); };
    if (first0 <= pos) attend(first0);
#pragma nounroll
    for (uint32_t first = first0; first <= pos && (first += step) <= pos;) {
        load(first);
        kv.lay_down(sh->ct[wave], lane);
        attend(first);
    }
    if (wave < a.attend) pb_leave(sh->merge, run, group, wave, lane);
    __syncthreads();
    float mean = 0.f;
    if (!pb_parts(a, sh->merge, kvh, split, group, s.vdim, base + PB_T_REC, recs, mean, cx)) return false;
    if (split > 0) return true;
    const float y = mean * sh->raw[min(gv + tid, ne - 1)], other = lane_xor<1>(y);
    if (tid < group * s.vdim && !(tid & 1u)) stc64(a.tout + (kvh * group * s.vdim + tid) / 2, base + PB_T_OUT, pb_pack(y, other));
    if (a.stamps && role == 0 && tid == 0) a.stamps[5 * l + 2] = wall_clock64();
    return true;
}

// ---- linear attention: a workgroup per head -------------------------------------------------------------------------------------------
// [decay | state, read-out | norm * gate].  The state of position p is in half p % 2 of the buffer: a step that is given up leaves its own untouched.
template <uint32_t WAVES>
struct PbLinear {
    static constexpr int STATE = PB_STATE * PB_WAVES / WAVES <= 8 ? PB_STATE * PB_WAVES / WAVES : 8;
    static constexpr uint32_t THREADS = WAVES * 64;
    v4f st[STATE];
    float w2[PB_LOW], b2, nw[PB_LVDIM / 64];
    // what a head's step reads that no other workgroup makes
    __device__ __forceinline__ void load(const PbArgs& a, const PbLayer& L, uint32_t head, uint32_t pos, uint32_t tid, uint32_t lane) {
        const LinearShape& s = a.ns;
        const uint32_t cols = s.vdim / 4, groups = THREADS / cols, rg = tid / cols, c = tid - rg * cols;
        const float* from = reinterpret_cast<float*>(pb_ptr(L.cache)) + (size_t)(pos & 1u) * s.state() + (size_t)head * s.dim * s.vdim;
#pragma unroll
        for (uint32_t i = 0; i < (uint32_t)STATE; i++)
            st[i] = __builtin_bit_cast(v4f, ldg(reinterpret_cast<const uint4*>(from + min(rg + i * groups, s.dim - 1) * s.vdim + 4 * c)));
        const float* w = pb_ptr(L.wa);
        const uint32_t ch = head * s.dim + min(tid, s.dim - 1);
        b2 = pb_f32(pb_ptr(L.wb), ch);
#pragma unroll
        for (uint32_t r = 0; r < PB_LOW; r++) w2[r] = pb_f32(w, min(r, s.rank - 1) * s.qk() + ch);
#pragma unroll
        for (uint32_t i = 0; i < PB_LVDIM / 64; i++) nw[i] = pb_f32(pb_ptr(L.wc), min(lane + 64 * i, s.vdim - 1));
    }
};
template <uint32_t WAVES>
__device__ __forceinline__ bool pb_linear_layer(const PbArgs& a, const PbLayer& L, PbLinear<WAVES>& in, PbLinearLds<WAVES>* sh, uint32_t head, uint32_t l, uint32_t pos, PollCtx& cx) {
    constexpr int STATE = PbLinear<WAVES>::STATE;
    const LinearShape& s = a.ns;
    const uint32_t lane = cx.lane, wave = cx.wave, tid = cx.tid, base = a.tag_base + l * PB_TAGS;
    const uint32_t cols = s.vdim / 4, groups = PbLinear<WAVES>::THREADS / cols, rg = tid / cols, c = tid - rg * cols;      // cols divides the wave
    float* to = reinterpret_cast<float*>(pb_ptr(L.cache)) + (size_t)((pos + 1) & 1u) * s.state() + (size_t)head * s.dim * s.vdim;
    v4f (&st)[STATE] = in.st;
    float (&w2)[PB_LOW] = in.w2, (&nw)[PB_LVDIM / 64] = in.nw;
    const float b2 = in.b2;
    // q, k, v, gate, low
    const uint32_t e1 = s.dim, e2 = 2 * s.dim, e3 = e2 + s.vdim, e4 = e3 + s.vdim, ne = e4 + s.rank;
    if (wave < PB_POLL) {
        constexpr int N = 2;
        static_assert(2 * 64 + 2 * PB_LVDIM + PB_LOW <= N * PB_POLL_THREADS, "fetched at once");
        uint32_t v[N];
        auto at = [&](uint32_t e) {
            const uint32_t v0 = 2 * s.qk(), low = v0 + s.heads * s.vdim, g0 = s.raw_row();
            return a.traw + (e < e1 ? head * s.dim + e : e < e2 ? s.qk() + head * s.dim + (e - e1) : e < e3 ? v0 + head * s.vdim + (e - e2) : e < e4 ? g0 + head * s.vdim + (e - e3) : low + (e - e4));
        };
        poll_tagged<N>([&](int i) { return at(min(cx.tid + i * PB_POLL_THREADS, ne - 1)); }, [&](int) { return base + PB_T_RAW; }, v, cx);
#pragma unroll
        for (int i = 0; i < N; i++)
            if (cx.tid + i * PB_POLL_THREADS < ne) sh->raw[cx.tid + i * PB_POLL_THREADS] = __uint_as_float(v[i]);
    }
    __syncthreads();
    if (*cx.sh_abort) return false;
    if (tid < s.dim) {
        float z = b2;
#pragma unroll
        for (uint32_t r = 0; r < PB_LOW; r++)
            if (r < s.rank) z = fmaf(w2[r], sh->raw[e4 + r], z);
        // sigmoid(z)^(1 / tau), with log sigmoid(z) = min(z, 0) - log(1 + e^-|z|)
        sh->a[tid] = expf((fminf(z, 0.f) - log1pf(expf(-fabsf(z)))) * s.inv_tau);
    }
    __syncthreads();
    v4f acc = (v4f){0.f, 0.f, 0.f, 0.f};
    const v4f v = *reinterpret_cast<const v4f*>(sh->raw + e2 + 4 * c);
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)STATE; i++) {
        const uint32_t d = rg + i * groups;
        if (d < s.dim) {
            const float dec = sh->a[d], k = sh->raw[e1 + d], q = sh->raw[d] * s.q_scale;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                st[i][j] = fmaf(dec, st[i][j], k * v[j]);
                acc[j] = fmaf(q, st[i][j], acc[j]);
            }
        }
    }
    // lanes of a wave that share a column are `cols` apart
#pragma unroll
    for (int j = 0; j < 4; j++) {
        if (cols <= 8) acc[j] = lane_xor_add<8>(acc[j]);
        if (cols <= 16) acc[j] = lane_xor_add<16>(acc[j]);
        if (cols <= 32) acc[j] = lane_xor_add<32>(acc[j]);
    }
    if (lane < cols) sh->part[wave][lane] = acc;
    __syncthreads();
    if (wave == 0) {
        float o[PB_LVDIM / 64], ss = 0.f;
#pragma unroll
        for (uint32_t i = 0; i < PB_LVDIM / 64; i++) {
            const uint32_t e = lane + 64 * i;
            o[i] = 0.f;
            if (e < s.vdim) {
#pragma unroll
                for (uint32_t w = 0; w < WAVES; w++) o[i] += reinterpret_cast<const float*>(sh->part[w])[e];
            }
            ss = fmaf(o[i], o[i], ss);                                // zero past vdim_n
        }
        const float inv = 1.0f / sqrtf(wave_sum(ss) / (float)s.vdim_n + s.eps);
#pragma unroll
        for (uint32_t i = 0; i < PB_LVDIM / 64; i++) {
            const uint32_t e = lane + 64 * i;
            if (e < s.vdim) stc64(a.tout + head * s.vdim + e, base + PB_T_OUT, __float_as_uint(o[i] * inv * nw[i] * sh->raw[e3 + e]));
        }
        if (a.stamps && head == 0 && lane == 0) a.stamps[5 * l + 2] = wall_clock64();
    }
    // the state is the next step's
#pragma unroll
    for (uint32_t i = 0; i < (uint32_t)STATE; i++) {
        const uint32_t d = rg + i * groups;
        if (d < s.dim) stg(reinterpret_cast<uint4*>(to + d * s.vdim + 4 * c), __builtin_bit_cast(uint4, st[i]));
    }
    return true;
}

// The logits of a tile of 16 rows and the best of them; every column is the same: lane l holds rows 4 (l / 16) .. + 3.
__device__ __forceinline__ void pb_logits(const PbArgs& a, uint32_t tile, const v4f& acc, uint32_t lane, ArgPair& best) {
#pragma unroll
    for (uint32_t r = 0; r < 4; r++) {
        const uint32_t row = tile * 16 + 4 * (lane >> 4) + r;
        if (row >= a.head.N || (lane & 15u) != r) continue;
        float v = acc[r];
        if (a.cap > 0.f) v = a.cap * tanhf(v / a.cap);
        stg(a.logits + row, v);
        // apply_repeat_penalty (project.rs:505-513) ahead of the argmax.  The lane that holds the row of the token being fed is the only one in the grid to touch
        // that counter: it adds this step's occurrence.
        if (a.penalty > 1.0f) {
            const bool fed = row == a.token;
            const uint32_t n = ldg(a.counts + row) + (fed ? 1u : 0u);
            if (fed) { stg(a.counts + row, n); stg(a.state + 4, a.step_seq); }      // so that a step that gives up later can be undone
            v = repeat_penalised(v, n, a.penalty);
        }
        best = arg_better(best, ArgPair{v, row});
    }
}
// The grid's best, by its first workgroup; the step's end.
__device__ __forceinline__ void pb_choose(const PbArgs& a, ArgPair best, ArgPair* sh_arg, uint32_t pos, PollCtx& cx) {
    const uint32_t th = a.tag_base + a.L * PB_TAGS, T = gridDim.x;
    auto stamp = [&](uint32_t slot) {
        if (a.stamps && cx.wg == 0 && cx.tid == 0) a.stamps[slot] = wall_clock64();
    };
    best = best_of_workgroup<PB_WAVES>(best, sh_arg, cx);
    if (cx.tid == 0) {
        stc64(a.tpart + 2 * cx.wg, th, __float_as_uint(best.v));
        stc64(a.tpart + 2 * cx.wg + 1, th, best.i);
    }
    stamp(5 * a.L + 1);
    if (cx.wg != 0) return;
    ArgPair p{-INFINITY, 0};
    for (uint32_t w = cx.tid; w < T; w += PB_THREADS) {
        uint32_t v[2];
        poll_tagged<2>([&](int i) { return a.tpart + 2 * w + (uint32_t)i; }, [&](int) { return th; }, v, cx);
        p = arg_better(p, ArgPair{__uint_as_float(v[0]), v[1]});
    }
    p = best_of_workgroup<PB_WAVES>(p, sh_arg, cx);
    if (*cx.sh_abort) return;
    if (cx.tid == 0) {
        a.state[2] = p.i;
        a.state[1] = p.i;
        a.state[0] = pos + 1;
        if (!(a.penalty > 1.0f)) a.counts[a.token] += 1;          // nobody read the counters in this launch
        stamp(5 * a.L + 2);
        // the host may be spinning on this word instead of waiting for the stream
        if (a.host_out) __hip_atomic_store(a.host_out, ((unsigned long long)a.host_seq << 32) | p.i, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

// ---- the kernel ---------------------------------------------------------------------------------------------------------------------------
// LATENT: elementwise norms, latent attention; else layer norms, linear and grouped attention.
template <bool LATENT>
__global__ __launch_bounds__(PB_THREADS) void decode_block_kernel(PbArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ uint32_t sh_abort;
    __shared__ ArgPair sh_arg[PB_WAVES];
    __bf16* const vec = reinterpret_cast<__bf16*>(smem);
    float* const red = reinterpret_cast<float*>(smem + a.off_red);                // [tile][wave][16 rows]
    float* const stats = reinterpret_cast<float*>(smem + a.off_stats);            // [wave][mean, sum of squares around it]
    const PbLayer* layers = reinterpret_cast<const PbLayer*>(smem + a.off_layers);
    typedef std::conditional_t<LATENT, PbLatentLds, PbKakiraxLds<PB_WAVES>> AttnLds;
    AttnLds* attn = reinterpret_cast<AttnLds*>(smem + a.off_attn);
    float* recs;                              // parts of other workgroups: where the transposed values are, when those are done with
    if constexpr (LATENT) recs = reinterpret_cast<float*>(attn->ct);
    else recs = reinterpret_cast<float*>(attn->grouped.ct);

    PollCtx cx;
    cx.tid = threadIdx.x;
    cx.lane = threadIdx.x & 63u;
    cx.wave = pb_sgpr(threadIdx.x >> 6);
    cx.wg = blockIdx.x;
    cx.G = a.G;
    cx.spin_limit = a.spin_limit;
    cx.sh_abort = &sh_abort;
    cx.abort_flag = a.state + 3;
    const bool comp = cx.wave >= PB_POLL;
    const uint32_t c = comp ? cx.wave - PB_POLL : 0u;
    if (cx.tid == 0) sh_abort = 0;
    for (uint32_t i = cx.tid; i < a.plane * 2; i += PB_THREADS) reinterpret_cast<uint32_t*>(smem)[i] = 0;      // 4 planes of 2 bytes
    for (uint32_t i = cx.tid; i < a.L * (uint32_t)(sizeof(PbLayer) / 4); i += PB_THREADS) reinterpret_cast<uint32_t*>(smem + a.off_layers)[i] = ldg(reinterpret_cast<const uint32_t*>(a.layers) + i);
    if constexpr (LATENT) {
        for (uint32_t i = cx.tid; i < (4 * PB_QR + PB_DIM + 2 * PB_ROW) / 2; i += PB_THREADS) reinterpret_cast<uint32_t*>(attn->x)[i] = 0;
    } else {
        for (uint32_t i = cx.tid; i < sizeof(attn->grouped.q) / 4; i += PB_THREADS) reinterpret_cast<uint32_t*>(attn->grouped.q)[i] = 0;
    }
    const uint32_t pos = pb_sgpr(a.state[0]);
    __syncthreads();

    // A phase ends, and the next one begins, where the first workgroup with a part of it has handed that on.
    auto stamp = [&](uint32_t slot) {
        if (a.stamps && cx.wg == 0 && cx.tid == 0) a.stamps[slot] = wall_clock64();
    };
    // this lane's column of the vector; exact in bfloat16: every column the first plane
    const __bf16* const x1 = vec + 8 * (cx.lane >> 4);
    const __bf16* const x3 = x1 + (cx.lane & 3u) * a.plane;
    const __bf16* const zeros = x1 + 3 * a.plane;
    const PbMat mh = a.head;
    const uint32_t T = gridDim.x, WAVES = PB_COMP * T, lwv = c * T + cx.wg, chunks = (mh.K / 32 + PB_HEAD_U - 1) / PB_HEAD_U;
    // The output matrix: a wave's tiles, a set of pieces at a time.
    struct Cur { uint32_t tile, chunk; };
    auto next_of = [&](Cur u) { return u.chunk + 1 < chunks ? Cur{u.tile, u.chunk + 1} : Cur{u.tile + WAVES, 0u}; };
    auto head_load = [&](PbSet<1, PB_HEAD_U>& w, Cur u) {
        if (u.tile >= mh.tiles) return;
        const uint32_t at = min(u.tile * 16 + (cx.lane & 15u), mh.N - 1) * mh.K * 2 + (cx.lane >> 4) * 16, last = mh.K / 32 - 1;
#pragma unroll
        for (int i = 0; i < PB_HEAD_U; i++) w.f[0][i] = pb_load8(a.head_w, at + min(u.chunk * PB_HEAD_U + i, last) * 64);
    };
    PbSet<1, PB_HEAD_U> wh[2];
    const Cur u0{lwv, 0}, u1 = next_of(u0);

    // A vector from 32-bit elements of the stream, layer-normed on the way (N, as the sequence has it: mean, then squares around it); three planes, or rounded to the first.  Every wave
    // takes part in the barrier in the middle.
    constexpr int NX = PB_WIDTH / PB_POLL_THREADS;
    auto layer_norm_fetch = [&](const uint64_t* t, uint32_t tag, const float* w, bool planes) {
        float nw[NX], nb[NX], x[NX];
#pragma unroll
        for (int i = 0; i < NX; i++) {
            const uint32_t e = min(cx.tid + i * PB_POLL_THREADS, a.W - 1);
            nw[i] = pb_f32(w, e);
            nb[i] = pb_f32(w, a.W + e);
        }
        if (!tag) {
#pragma unroll
            for (int i = 0; i < NX; i++) x[i] = pb_embed(a, min(cx.tid + i * PB_POLL_THREADS, a.W - 1));
        } else {
            uint32_t v[NX];
            poll_tagged<NX>([&](int i) { return t + min(cx.tid + i * PB_POLL_THREADS, a.W - 1); }, [&](int) { return tag; }, v, cx);
#pragma unroll
            for (int i = 0; i < NX; i++) x[i] = __uint_as_float(v[i]);
        }
        // a wave's mean and squares around it, then the workgroup's from those: as exact as one mean for all
        float sum = 0.f;
        uint32_t mine = 0;
#pragma unroll
        for (int i = 0; i < NX; i++) {
            const uint32_t e0 = 64 * cx.wave + i * PB_POLL_THREADS;
            if (e0 + cx.lane < a.Wn) sum += x[i];
            mine += e0 < a.Wn ? min(64u, a.Wn - e0) : 0u;
        }
        const float n = (float)mine, mean_w = n > 0.f ? wave_sum(sum) / n : 0.f;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NX; i++) {
            const float d = x[i] - mean_w;
            if (cx.tid + i * PB_POLL_THREADS < a.Wn) ss = fmaf(d, d, ss);
        }
        ss = wave_sum(ss);
        if (cx.lane == 0) { stats[3 * cx.wave] = n; stats[3 * cx.wave + 1] = mean_w; stats[3 * cx.wave + 2] = ss; }
        __syncthreads();
        float mean = 0.f, sq = 0.f;
#pragma unroll
        for (uint32_t i = 0; i < PB_POLL; i++) mean = fmaf(stats[3 * i], stats[3 * i + 1], mean);
        mean /= (float)a.Wn;
#pragma unroll
        for (uint32_t i = 0; i < PB_POLL; i++) { const float d = stats[3 * i + 1] - mean; sq += fmaf(stats[3 * i] * d, d, stats[3 * i + 2]); }
        const float inv = 1.0f / sqrtf(sq / (float)a.Wn + a.eps);
#pragma unroll
        for (int i = 0; i < NX; i++) {
            const uint32_t e = cx.tid + i * PB_POLL_THREADS;
            if (e >= a.W) continue;
            const float y = (x[i] - mean) * inv * nw[i] + nb[i];
            if (planes) pb_put(vec, a.plane, e, y);
            else vec[e] = (__bf16)y;
        }
    };
    auto layer_norm_join = [&]() { if constexpr (!LATENT) __syncthreads(); };      // the computing waves' part of it
    constexpr int NP = (PB_WIDTH / 2 + PB_POLL_THREADS - 1) / PB_POLL_THREADS;     // pairs of a row of the stream a thread
    // A wave's results of T tiles into `red`, and a row's sum.
    auto leave = [&](v4f v, uint32_t t, bool planes) {
        if (planes) v = pb_columns(v);
        if ((cx.lane & 15u) == 0) *reinterpret_cast<v4f*>(red + (t * PB_COMP + c) * 16 + 4 * (cx.lane >> 4)) = v;
    };
    auto row_sum = [&](uint32_t r) {
        const float* p = red + (r >> 4) * PB_COMP * 16 + (r & 15u);
        float s = 0.f;
#pragma unroll
        for (uint32_t i = 0; i < PB_COMP; i++) s += p[16 * i];
        return s;
    };

    if (cx.wg < a.G) {
        const bool on_o = cx.wg * 16 < a.W, on_g = cx.wg * a.gate_up.T < a.gate_up.tiles;      // the workgroup's rows of the stream: one tile, o's and down's and the loop's
        if (!comp) {
            // the first wave finishes rows
            const uint32_t xrow = min(cx.wg * 16 + (cx.lane & 15u), a.W - 1);
            const bool mine = on_o && cx.lane < 16;
            float x = pb_embed(a, xrow);
#pragma nounroll
            for (uint32_t l = 0; l < a.L; l++) {
                asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
                const PbLayer& L = layers[l];
                const uint32_t base = a.tag_base + l * PB_TAGS, kind = pb_sgpr(L.kind), loop = LATENT ? pb_sgpr(L.loop) : 0u;
                const uint32_t x_in = l ? base - PB_TAGS + PB_T_DOWN : 0u;
                const PbMat mi = pb_of(a.in, kind);
                const bool on_i = cx.wg * mi.T < mi.tiles;
                stamp(5 * l);
                // what the rows' ends read
                float pw1 = 0.f, pb1 = 0.f, nw2 = 0.f, nb2 = 0.f, pw2 = 0.f, pb2 = 0.f, nwn = 0.f, nbn = 0.f;
                if constexpr (LATENT) {
                    if (cx.wave == 0) {
                        const float *p1 = pb_ptr(L.post1), *n2 = pb_ptr(L.norm2), *p2 = pb_ptr(L.post2), *nx = pb_ptr(L.next) ? pb_ptr(L.next) : n2;
                        pw1 = pb_f32(p1, xrow); pb1 = pb_f32(p1, a.W + xrow); nw2 = pb_f32(n2, xrow); nb2 = pb_f32(n2, a.W + xrow);
                        pw2 = pb_f32(p2, xrow); pb2 = pb_f32(p2, a.W + xrow); nwn = pb_f32(nx, xrow); nbn = pb_f32(nx, a.W + xrow);
                    }
                }
                // the stream's rows, `h` of them as the next product's input
                auto hand_on = [&](uint64_t* to, uint32_t tag, float h) {
                    if constexpr (LATENT) {
                        const float other = lane_xor<1>(h);
                        if (mine && !(cx.lane & 1u)) stc64(to + xrow / 2, tag, pb_pack(h, other));
                    } else {
                        if (mine) stc64(to + xrow, tag, __float_as_uint(h));
                    }
                };
                if constexpr (LATENT) {
                    if (loop && on_o) {
                        // [stream; embedding row], both as the sequence stores them
                        uint32_t* half = reinterpret_cast<uint32_t*>(vec) + a.W / 2;
                        for (uint32_t e = cx.tid; e < a.W / 2; e += PB_POLL_THREADS) half[e] = pb_pack(pb_embed(a, 2 * e), pb_embed(a, 2 * e + 1));
                        if (x_in) pb_fetch_pairs<NP>(a.th, x_in, a.W / 2, a.W / 2, reinterpret_cast<uint32_t*>(vec), cx);
                        else
                            for (uint32_t e = cx.tid; e < a.W / 2; e += PB_POLL_THREADS) reinterpret_cast<uint32_t*>(vec)[e] = pb_pack(pb_embed(a, 2 * e), pb_embed(a, 2 * e + 1));
                        __syncthreads();
                        if (sh_abort) return;
                        __syncthreads();
                        if (cx.wave == 0) {
                            x = row_sum(cx.lane & 15u);
                            const float* n1 = pb_ptr(L.norm1);
                            hand_on(a.tl, base + PB_T_LOOP, pb_tanh(L.alpha1, x, pb_f32(n1, xrow), pb_f32(n1, a.W + xrow)));
                        }
                    }
                }
                // ---- input product
                if (on_i) {
                    if constexpr (LATENT) {
                        if (loop || x_in) {
                            pb_fetch_pairs<NP>(loop ? a.tl : a.th, loop ? base + PB_T_LOOP : x_in, a.W / 2, a.W / 2, reinterpret_cast<uint32_t*>(vec), cx);
                        } else {
                            const float* n1 = pb_ptr(L.norm1);
                            for (uint32_t e = cx.tid; e < a.W; e += PB_POLL_THREADS) vec[e] = (__bf16)pb_tanh(L.alpha1, pb_embed(a, e), pb_f32(n1, e), pb_f32(n1, a.W + e));
                        }
                    } else {
                        layer_norm_fetch(a.th, x_in, pb_ptr(L.norm1), true);
                    }
                    __syncthreads();
                    if (sh_abort) return;
                    __syncthreads();
                    if (cx.wave == 0) {
                        const uint32_t n = 16 * mi.T, row = cx.wg * n + cx.lane, raw = LATENT ? a.ls.raw_row() : kind == PB_FIRST ? a.ns.raw_row() : a.gs.raw_row();
                        float v = row_sum(min(cx.lane, n - 1));
                        const float g = !LATENT && kind == PB_FIRST ? silu_f(v) : sigmoid_f(v);
                        if (row >= raw) v = (float)(__bf16)g;
                        if (cx.lane < n && row < mi.N) stc64(a.traw + row, base + PB_T_RAW, __float_as_uint(v));
                    }
                }
                stamp(5 * l + 1);
                // ---- output product
                if (on_o) {
                    const PbMat mo = pb_of(a.o, kind);
                    uint32_t* plane = reinterpret_cast<uint32_t*>(vec);
                    if (LATENT) pb_fetch_pairs<NP>(a.tout, base + PB_T_OUT, a.ls.heads * a.ls.vdim / 2, mo.K / 2, plane, cx);
                    else if (kind == PB_GROUPED) pb_fetch_pairs<NP>(a.tout, base + PB_T_OUT, a.gs.heads * a.gs.vdim / 2, mo.K / 2, plane, cx);
                    else pb_fetch_floats<NX>(a.tout, base + PB_T_OUT, a.ns.heads * a.ns.vdim, mo.K, vec, a.plane, cx);
                    __syncthreads();
                    if (sh_abort) return;
                    __syncthreads();
                    if (cx.wave == 0) {
                        const float v = row_sum(cx.lane & 15u);
                        x = LATENT ? pb_tanh(L.post_alpha1, v, pw1, pb1) + x : v + x;
                        hand_on(a.th, base + PB_T_O, LATENT ? pb_tanh(L.alpha2, x, nw2, nb2) : x);
                    }
                }
                stamp(5 * l + 3);
                // ---- gate;up
                if (on_g) {
                    if constexpr (LATENT) pb_fetch_pairs<NP>(a.th, base + PB_T_O, a.W / 2, a.W / 2, reinterpret_cast<uint32_t*>(vec), cx);
                    else layer_norm_fetch(a.th, base + PB_T_O, pb_ptr(L.norm2), true);
                    __syncthreads();
                    if (sh_abort) return;
                    __syncthreads();
                    if (cx.wave == 0) {
                        // rows 2 i and 2 i + 1 are gate and up of element i; four rows to a pair
                        const uint32_t n = 16 * a.gate_up.T, row = cx.wg * n + cx.lane;
                        const float v = row_sum(min(cx.lane, n - 1)), up = lane_xor<1>(v);
                        const float y = act_f((Act)a.act, v) * up, y1 = lane_xor<2>(y);
                        if (cx.lane < n && !(cx.lane & 3u) && row < a.gate_up.N) stc64(a.tact + row / 4, base + PB_T_ACT, pb_pack(y, y1));
                    }
                }
                stamp(5 * l + 4);
                // ---- down
                if (on_o) {
                    constexpr int N = PB_FF / 2 / PB_POLL_THREADS;
                    pb_fetch_pairs<N>(a.tact, base + PB_T_ACT, a.ff / 2, a.ff / 2, reinterpret_cast<uint32_t*>(vec), cx);
                    __syncthreads();
                    if (sh_abort) return;
                    __syncthreads();
                    if (cx.wave == 0) {
                        const float v = row_sum(cx.lane & 15u);
                        x = LATENT ? pb_tanh(L.post_alpha2, v, pw2, pb2) + x : v + x;
                        hand_on(a.th, base + PB_T_DOWN, LATENT && pb_ptr(L.next) ? pb_tanh(L.next_alpha, x, nwn, nbn) : x);
                    }
                }
            }
        } else {
            PbSet<PB_TI, PB_UI> wi;
            PbSet<1, PB_UO> wo;
            PbSet<PB_TG, PB_UI> wg;
            PbSet<1, PB_UD> wd;
            pb_load(wi, pb_ptr(layers[0].in), pb_of(a.in, pb_sgpr(layers[0].kind)), cx.wg, c, cx.lane);
#pragma nounroll
            for (uint32_t l = 0; l < a.L; l++) {
                asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
                const PbLayer& L = layers[l];
                const uint32_t kind = pb_sgpr(L.kind);
                const PbMat mi = pb_of(a.in, kind), mo = pb_of(a.o, kind);
                if constexpr (LATENT) {
                    if (pb_sgpr(L.loop) && on_o) {
                        PbSet<1, PB_UL> wl;
                        pb_load(wl, a.loop_w, a.loop, cx.wg, c, cx.lane);
                        __syncthreads();
                        if (sh_abort) return;
                        v4f acc[1];
                        pb_mul(wl, a.loop, c, x1, zeros, acc);
                        leave(acc[0], 0, false);
                        __syncthreads();
                    }
                }
                if (cx.wg * mi.T < mi.tiles) {
                    layer_norm_join();
                    __syncthreads();
                    if (sh_abort) return;
                    v4f acc[PB_TI];
                    pb_mul(wi, mi, c, LATENT ? x1 : x3, zeros, acc);
#pragma unroll
                    for (int t = 0; t < PB_TI; t++) leave(acc[t], t, !LATENT);
                    __syncthreads();
                }
                // While the attention is at work nothing else is on its way to this workgroup.
                pb_load(wo, pb_ptr(L.o), mo, cx.wg, c, cx.lane);
                pb_load(wg, pb_ptr(L.gate_up), a.gate_up, cx.wg, c, cx.lane);
                pb_load(wd, pb_ptr(L.down), a.down, cx.wg, c, cx.lane);
                {
                    const PbLayer& N = layers[min(l + 1, a.L - 1)];
                    pb_load(wi, pb_ptr(N.in), pb_of(a.in, pb_sgpr(N.kind)), cx.wg, c, cx.lane);
                }
                if (on_o) {
                    __syncthreads();
                    if (sh_abort) return;
                    const bool planes = !LATENT && kind == PB_FIRST;
                    v4f acc[1];
                    pb_mul(wo, mo, c, planes ? x3 : x1, zeros, acc);
                    leave(acc[0], 0, planes);
                    __syncthreads();
                }
                if (on_g) {
                    layer_norm_join();
                    __syncthreads();
                    if (sh_abort) return;
                    v4f acc[PB_TG];
                    pb_mul(wg, a.gate_up, c, LATENT ? x1 : x3, zeros, acc);
#pragma unroll
                    for (int t = 0; t < PB_TG; t++) leave(acc[t], t, !LATENT);
                    __syncthreads();
                }
                if (on_o) {
                    __syncthreads();
                    if (sh_abort) return;
                    v4f acc[1];
                    pb_mul(wd, a.down, c, x1, zeros, acc);
                    leave(acc[0], 0, false);
                    __syncthreads();
                }
            }
            head_load(wh[0], u0);
        }
    } else {
        const uint32_t role = cx.wg - a.G;
        if constexpr (LATENT) {
            if (role < a.ls.heads * a.splits && !pb_latent_layers(a, layers, attn, recs, pos, cx)) return;
        } else {
            const bool on_n = role < a.ns.heads, on_g = role < a.gs.kv_heads * a.splits;
#pragma nounroll
            for (uint32_t l = 0; (on_n || on_g) && l < a.L; l++) {
                asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
                if (pb_sgpr(layers[l].kind) == PB_FIRST) {
                    PbLinear<PB_WAVES> in;
                    if (on_n) in.load(a, layers[l], role, pos, cx.tid, cx.lane);
                    if (on_n && !pb_linear_layer(a, layers[l], in, &attn->linear, role, l, pos, cx)) return;
                } else if (on_g && !pb_grouped_layer<PB_WAVES>(a, layers[l], &attn->grouped, recs, role, l, pos, cx)) {
                    return;
                }
            }
        }
        asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
        if (comp) head_load(wh[0], u0);
        // a workgroup without rows in the layers looks for the final row now and then only
        if (cx.tid == 0) {
            uint32_t spins = 0;
            while ((uint32_t)(ldc64(a.th + (LATENT ? a.W / 2 : a.W) - 1) >> 32) != a.tag_base + (a.L - 1) * PB_TAGS + PB_T_DOWN && ++spins <= cx.spin_limit &&
                   ((spins & 255u) != 0 || __hip_atomic_load(cx.abort_flag, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) == 0))
                __builtin_amdgcn_s_sleep(16);
        }
        __syncthreads();
    }

    // ---- final norm | output matrix | argmax
    asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
    stamp(5 * a.L);
    ArgPair best{-INFINITY, 0};
    const uint32_t x_last = a.tag_base + (a.L - 1) * PB_TAGS + PB_T_DOWN;
    if (!comp) {
        if constexpr (LATENT) pb_fetch_pairs<NP>(a.th, x_last, a.W / 2, a.W / 2, reinterpret_cast<uint32_t*>(vec), cx);
        else layer_norm_fetch(a.th, x_last, a.final_norm, false);
        __syncthreads();
        if (sh_abort) return;
    } else {
        layer_norm_join();
        __syncthreads();
        if (sh_abort) return;
        v4f acc = (v4f){0.f, 0.f, 0.f, 0.f};
        auto work = [&](const PbSet<1, PB_HEAD_U>& w, Cur u) {
#pragma unroll
            for (int i = 0; i < PB_HEAD_U; i++) {
                const uint32_t k = u.chunk * PB_HEAD_U + i;
                acc = mma16(w.f[0][i], load8(k < mh.K / 32 ? x1 + 32 * k : zeros), acc);
            }
            if (u.chunk + 1 < chunks) return;
            pb_logits(a, u.tile, acc, cx.lane, best);
            acc = (v4f){0.f, 0.f, 0.f, 0.f};
        };
        head_load(wh[1], u1);
        for (Cur u = u0, v = u1; u.tile < mh.tiles;) {
            work(wh[0], u);
            u = next_of(v);
            head_load(wh[0], u);
            if (v.tile >= mh.tiles) break;
            work(wh[1], v);
            v = next_of(u);
            head_load(wh[1], v);
        }
    }
    pb_choose(a, best, sh_arg, pos, cx);
}

// ---- the wide form ------------------------------------------------------------------------------------------------------------------------
// Layers that registers cannot hold (linear and grouped attention): every workgroup streams its rows of every matrix, and the heads are the polling waves' of as many workgroups.  A tile is
// 8 rows by two halves of the depth (row r of the product: row r % 8, half r / 8), tile t of a workgroup the grid's tile t G + wg: no row of a 2048-row matrix is left over on 256 workgroups.  A
// column of the vector is a plane of one half.
//
// Per token in us, kernel sequence / this, kakirax_1b (width 2048, feed-forward 8192, three layers of linear attention to one of grouped): 20 rows 837 / 701, 902 838 / 712, 2400 839 / 723,
// 6000 845 / 738.  What bounds it: the weights (134 MB a layer, 24 us of its 38) and the hand-overs while nothing is on its way (8 us between down's vector and the next input product's, 5 in
// the others).  A compute unit takes about 64 KB of requests and a wave that has more to ask for stands still, so what decided the form is what stands in front of a barrier (us a token):
//   * a head's workgroup asks for its next input product only when it has its output product (its polls would wait behind 260 KB): 760 -> 753, and its barriers come first: 753 -> 722;
//   * down is requested behind the barrier that ends gate;up, not ahead of it: 753 -> 721;
//   * the next layer's input product goes into LDS while the heads are at work, for which registers have no room: the same time, but no spills with half of gate;up early as well.
// Without effect: at most 4, 8 or 12 KB of a wave under way, output product and a quarter of gate;up requested a phase earlier (720).  Spilled registers cost more than anything: a spill waits for
// all loads (28 of them: 758 -> 840).
// Limits: the width (a fifth piece, 2560, spills 120 bytes a lane more) and gate;up's tiles (ten: 92 more) by registers; the depth of down is what the model at hand has (10240 spills nothing more).
constexpr uint32_t PW_WIDTH = 2048, PW_FF = 8192;
constexpr int PW_U = 4, PW_UD = 16;          // pieces of a wave in a half: depth PW_WIDTH, PW_FF
constexpr int PW_TI = 4, PW_TIL = 3, PW_TG = 8, PW_TGA = 4;      // tiles of a workgroup: input product (the first PW_TIL of them in LDS), gate;up (the first PW_TGA of them requested early)
static_assert(PW_TGA % 2 == 0 && PW_TG % 2 == 0, "tiles are worked in pairs");
constexpr uint32_t PW_SLOT = PW_TIL * PW_U * 1024;                   // LDS of a wave's pieces of an input product
constexpr int PW_HEAD_U = 8;

typedef __amdgpu_buffer_rsrc_t PwRsrc;
__device__ __forceinline__ PwRsrc pw_rsrc(const __bf16* w, const PbMat& m) { return __builtin_amdgcn_make_buffer_rsrc((void*)w, 0, m.N * m.K * 2, 0x00020000); }
// Tiles t0 .. t0 + T of a workgroup; rows past the matrix read as zero.
template <int T, int U>
__device__ __forceinline__ void pw_load(PbSet<T, U>& s, const __bf16* w, const PbMat& m, uint32_t t0, uint32_t G, uint32_t wg, uint32_t c, uint32_t lane) {
    asm volatile("" : "+v"(lane));
    __builtin_amdgcn_sched_barrier(0);
    const PwRsrc rsrc = pw_rsrc(w, m);
    const uint32_t last = m.K / 64 - 1;
#pragma unroll
    for (int t = 0; t < T; t++) {
        const uint32_t at = (((t0 + t) * G + wg) * 8 + (lane & 7u)) * m.K * 2 + ((lane >> 3) & 1u) * m.K + (lane >> 4) * 16;
#pragma unroll
        for (int i = 0; i < U; i++) s.f[t][i] = __builtin_bit_cast(v8bf, __builtin_amdgcn_raw_buffer_load_b128(rsrc, at, min(c * m.per + min((uint32_t)i, m.per - 1), last) * 64, 0));
    }
    __builtin_amdgcn_sched_barrier(0);
}
// The first PW_TIL tiles into the wave's LDS, a lane's 16 bytes of a piece where it reads them.
__device__ __forceinline__ void pw_load_lds(uint8_t* slot, const __bf16* w, const PbMat& m, uint32_t G, uint32_t wg, uint32_t c, uint32_t lane) {
    asm volatile("" : "+v"(lane));
    __builtin_amdgcn_sched_barrier(0);
    const PwRsrc rsrc = pw_rsrc(w, m);
    const uint32_t last = m.K / 64 - 1;
#pragma unroll
    for (int t = 0; t < PW_TIL; t++) {
        const uint32_t at = ((t * G + wg) * 8 + (lane & 7u)) * m.K * 2 + ((lane >> 3) & 1u) * m.K + (lane >> 4) * 16;
#pragma unroll
        for (int i = 0; i < PW_U; i++)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (__attribute__((address_space(3))) void*)(slot + (t * PW_U + i) * 1024), 16, at, min(c * m.per + min((uint32_t)i, m.per - 1), last) * 64, 0, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
}
template <int T, int U>
__device__ __forceinline__ void pw_mul(const PbSet<T, U>& s, const PbMat& m, uint32_t c, const __bf16* x, const __bf16* zeros, v4f (&acc)[T]) {
#pragma unroll
    for (int t = 0; t < T; t++) acc[t] = (v4f){0.f, 0.f, 0.f, 0.f};
    constexpr int B = T > 1 ? 2 : U < 8 ? U : 8;
#pragma unroll
    for (int i0 = 0; i0 < U; i0 += B) {
        v8bf b[B];
#pragma unroll
        for (int i = 0; i < B; i++) {
            const uint32_t k = c * m.per + i0 + i;
            b[i] = load8((uint32_t)(i0 + i) < m.per && k < m.K / 64 ? x + 32 * k : zeros);
        }
#pragma unroll
        for (int i = 0; i < B; i++)
#pragma unroll
            for (int t = 0; t < T; t++) acc[t] = mma16(s.f[t][i0 + i], b[i], acc[t]);
    }
}

typedef PbKakiraxLds<PB_POLL> PwAttnLds;

__global__ __launch_bounds__(PB_THREADS) void decode_block_wide_kernel(PbArgs a) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ uint32_t sh_abort;
    __shared__ ArgPair sh_arg[PB_WAVES];
    __bf16* const vec = reinterpret_cast<__bf16*>(smem);
    float* const red = reinterpret_cast<float*>(smem + a.off_red);                // [tile][wave][16 rows]
    float* const stats = reinterpret_cast<float*>(smem + a.off_stats);
    const PbLayer* layers = reinterpret_cast<const PbLayer*>(smem + a.off_layers);
    PwAttnLds* attn = reinterpret_cast<PwAttnLds*>(smem + a.off_attn);
    float* recs = reinterpret_cast<float*>(attn->grouped.ct);

    PollCtx cx;
    cx.tid = threadIdx.x;
    cx.lane = threadIdx.x & 63u;
    cx.wave = pb_sgpr(threadIdx.x >> 6);
    cx.wg = blockIdx.x;
    cx.G = a.G;
    cx.spin_limit = a.spin_limit;
    cx.sh_abort = &sh_abort;
    cx.abort_flag = a.state + 3;
    const bool comp = cx.wave >= PB_POLL;
    const uint32_t c = comp ? cx.wave - PB_POLL : 0u, G = a.G;
    if (cx.tid == 0) sh_abort = 0;
    for (uint32_t i = cx.tid; i < sizeof(attn->grouped.q) / 4; i += PB_THREADS) reinterpret_cast<uint32_t*>(attn->grouped.q)[i] = 0;
    __shared__ __align__(16) __bf16 sh_zeros[32];
    if (cx.tid < 32) sh_zeros[cx.tid] = (__bf16)0.0f;
    uint8_t* const slot = smem + a.off_in + c * PW_SLOT;
    for (uint32_t i = cx.tid; i < a.L * (uint32_t)(sizeof(PbLayer) / 4); i += PB_THREADS) reinterpret_cast<uint32_t*>(smem + a.off_layers)[i] = ldg(reinterpret_cast<const uint32_t*>(a.layers) + i);
    const uint32_t pos = pb_sgpr(a.state[0]);
    __syncthreads();

    auto stamp = [&](uint32_t slot) {
        if (a.stamps && cx.wg == 0 && cx.tid == 0) a.stamps[slot] = wall_clock64();
    };
    // this lane's column of a vector of K elements: a half of a plane
    auto column = [&](uint32_t K, bool planes) { return vec + (planes ? min((cx.lane >> 1) & 3u, 2u) * a.plane : 0u) + (cx.lane & 1u) * (K / 2) + 8 * (cx.lane >> 4); };
    const __bf16* const zeros = sh_zeros + 8 * (cx.lane >> 4);
    const PbMat mh = a.head;
    const uint32_t T = gridDim.x, WAVES = PB_COMP * T, lwv = c * T + cx.wg, chunks = (mh.K / 32 + PW_HEAD_U - 1) / PW_HEAD_U;
    struct Cur { uint32_t tile, chunk; };
    auto next_of = [&](Cur u) { return u.chunk + 1 < chunks ? Cur{u.tile, u.chunk + 1} : Cur{u.tile + WAVES, 0u}; };
    auto head_load = [&](PbSet<1, PW_HEAD_U>& w, Cur u) {
        if (u.tile >= mh.tiles) return;
        const uint32_t at = min(u.tile * 16 + (cx.lane & 15u), mh.N - 1) * mh.K * 2 + (cx.lane >> 4) * 16, last = mh.K / 32 - 1;
#pragma unroll
        for (int i = 0; i < PW_HEAD_U; i++) w.f[0][i] = pb_load8(a.head_w, at + min(u.chunk * PW_HEAD_U + i, last) * 64);
    };

    // As in the narrow form, twice: a wave's mean and squares around it, then the workgroup's.
    constexpr int NX = PW_WIDTH / PB_POLL_THREADS;
    auto layer_norm_fetch = [&](const uint64_t* t, uint32_t tag, const float* w, bool planes) {
        float nw[NX], nb[NX], x[NX];
#pragma unroll
        for (int i = 0; i < NX; i++) {
            const uint32_t e = min(cx.tid + i * PB_POLL_THREADS, a.W - 1);
            nw[i] = pb_f32(w, e);
            nb[i] = pb_f32(w, a.W + e);
        }
        if (!tag) {
#pragma unroll
            for (int i = 0; i < NX; i++) x[i] = pb_embed(a, min(cx.tid + i * PB_POLL_THREADS, a.W - 1));
        } else {
            uint32_t v[NX];
            poll_tagged<NX>([&](int i) { return t + min(cx.tid + i * PB_POLL_THREADS, a.W - 1); }, [&](int) { return tag; }, v, cx);
#pragma unroll
            for (int i = 0; i < NX; i++) x[i] = __uint_as_float(v[i]);
        }
        float sum = 0.f;
        uint32_t mine = 0;
#pragma unroll
        for (int i = 0; i < NX; i++) {
            const uint32_t e0 = 64 * cx.wave + i * PB_POLL_THREADS;
            if (e0 + cx.lane < a.Wn) sum += x[i];
            mine += e0 < a.Wn ? min(64u, a.Wn - e0) : 0u;
        }
        const float n = (float)mine, mean_w = n > 0.f ? wave_sum(sum) / n : 0.f;
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NX; i++) {
            const float d = x[i] - mean_w;
            if (cx.tid + i * PB_POLL_THREADS < a.Wn) ss = fmaf(d, d, ss);
        }
        ss = wave_sum(ss);
        if (cx.lane == 0) { stats[3 * cx.wave] = n; stats[3 * cx.wave + 1] = mean_w; stats[3 * cx.wave + 2] = ss; }
        __syncthreads();
        float mean = 0.f, sq = 0.f;
#pragma unroll
        for (uint32_t i = 0; i < PB_POLL; i++) mean = fmaf(stats[3 * i], stats[3 * i + 1], mean);
        mean /= (float)a.Wn;
#pragma unroll
        for (uint32_t i = 0; i < PB_POLL; i++) { const float d = stats[3 * i + 1] - mean; sq += fmaf(stats[3 * i] * d, d, stats[3 * i + 2]); }
        const float inv = 1.0f / sqrtf(sq / (float)a.Wn + a.eps);
#pragma unroll
        for (int i = 0; i < NX; i++) {
            const uint32_t e = cx.tid + i * PB_POLL_THREADS;
            if (e >= a.W) continue;
            const float y = (x[i] - mean) * inv * nw[i] + nb[i];
            if (planes) pb_put(vec, a.plane, e, y);
            else vec[e] = (__bf16)y;
        }
    };
    auto leave = [&](v4f v, uint32_t t, bool planes) {
        const uint32_t lg = cx.lane >> 4;
        if (planes) {
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = lane_xor_add<4>(lane_xor_add<2>((cx.lane & 6u) == 6u ? 0.f : v[r]));      // there is no fourth plane
        }
        if ((cx.lane & 15u) == lg >> 1) *reinterpret_cast<v4f*>(red + (t * PB_COMP + c) * 16 + 4 * lg) = v;
    };
    auto row_sum = [&](uint32_t t, uint32_t r) {
        const float* p = red + t * PB_COMP * 16 + r;
        float s = 0.f;
#pragma unroll
        for (uint32_t i = 0; i < PB_COMP; i++) s += p[16 * i] + p[16 * i + 8];
        return s;
    };
    const bool on_o = cx.wg * 8 < a.W, on_g = cx.wg < a.gate_up.tiles;
    const uint32_t grouped_roles = a.gs.kv_heads * a.splits;
    if (!comp) {
        const uint32_t sub = cx.lane & 7u, xrow = min(cx.wg * 8 + sub, a.W - 1);
        const bool mine = on_o && cx.lane < 8;
        float x = pb_embed(a, xrow);
        auto hand_on = [&](uint32_t tag, float v) {
            if (mine) stc64(a.th + xrow, tag, __float_as_uint(v));
        };
#pragma nounroll
        for (uint32_t l = 0; l < a.L; l++) {
            asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
            const PbLayer& L = layers[l];
            const uint32_t base = a.tag_base + l * PB_TAGS, kind = pb_sgpr(L.kind), x_in = l ? base - PB_TAGS + PB_T_DOWN : 0u;
            const PbMat mi = pb_of(a.in, kind), mo = pb_of(a.o, kind);
            stamp(5 * l);
            PbLinear<PB_POLL> lin;
            const bool on_n = kind == PB_FIRST && cx.wg < a.ns.heads, on_k = kind == PB_GROUPED && cx.wg < grouped_roles;
            if (on_n) lin.load(a, L, cx.wg, pos, cx.tid, cx.lane);
            if (cx.wg < mi.tiles) {
                layer_norm_fetch(a.th, x_in, pb_ptr(L.norm1), true);
                __syncthreads();
                if (sh_abort) return;
                __syncthreads();
                if (cx.wave == 0) {
                    const uint32_t t = cx.lane >> 3, row = (t * G + cx.wg) * 8 + sub, raw = kind == PB_FIRST ? a.ns.raw_row() : a.gs.raw_row();
                    float v = row_sum(min(t, mi.T - 1), sub);
                    const float g = kind == PB_FIRST ? silu_f(v) : sigmoid_f(v);
                    if (row >= raw) v = (float)(__bf16)g;
                    if (t < mi.T && row < mi.N) stc64(a.traw + row, base + PB_T_RAW, __float_as_uint(v));
                }
            }
            stamp(5 * l + 1);
            if (on_n) {
                if (!pb_linear_layer(a, L, lin, &attn->linear, cx.wg, l, pos, cx)) return;
            } else if (on_k) {
                if (!pb_grouped_layer<PB_POLL>(a, L, &attn->grouped, recs, cx.wg, l, pos, cx)) return;
            }
            // ---- output product
            if (on_o) {
                uint32_t* plane = reinterpret_cast<uint32_t*>(vec);
                if (kind == PB_GROUPED) pb_fetch_pairs<NX / 2>(a.tout, base + PB_T_OUT, a.gs.heads * a.gs.vdim / 2, mo.K / 2, plane, cx);
                else pb_fetch_floats<NX>(a.tout, base + PB_T_OUT, a.ns.heads * a.ns.vdim, mo.K, vec, a.plane, cx);
                __syncthreads();
                if (sh_abort) return;
                __syncthreads();
                if (cx.wave == 0) {
                    x += row_sum(0, sub);
                    hand_on(base + PB_T_O, x);
                }
            }
            stamp(5 * l + 3);
            // ---- gate;up
            if (on_g) {
                layer_norm_fetch(a.th, base + PB_T_O, pb_ptr(L.norm2), true);
                __syncthreads();
                if (sh_abort) return;
                __syncthreads();
                if (cx.wave == 0) {
                    // rows 2 i and 2 i + 1 are gate and up of element i; four rows to a pair
                    const uint32_t t = cx.lane >> 3, row = (t * G + cx.wg) * 8 + sub;
                    const float v = row_sum(min(t, a.gate_up.T - 1), sub), up = lane_xor<1>(v);
                    const float y = act_f((Act)a.act, v) * up, y1 = lane_xor<2>(y);
                    if (t < a.gate_up.T && !(cx.lane & 3u) && row < a.gate_up.N) stc64(a.tact + row / 4, base + PB_T_ACT, pb_pack(y, y1));
                }
            }
            stamp(5 * l + 4);
            // ---- down
            if (on_o) {
                constexpr int N = PW_FF / 2 / PB_POLL_THREADS;
                pb_fetch_pairs<N>(a.tact, base + PB_T_ACT, a.ff / 2, a.ff / 2, reinterpret_cast<uint32_t*>(vec), cx);
                __syncthreads();
                if (sh_abort) return;
                __syncthreads();
                if (cx.wave == 0) {
                    x += row_sum(0, sub);
                    hand_on(base + PB_T_DOWN, x);
                }
            }
        }
    } else {
        PbSet<PW_TI - PW_TIL, PW_U> wi;      // the input product's tiles behind those in LDS
        pw_load_lds(slot, pb_ptr(layers[0].in), pb_of(a.in, pb_sgpr(layers[0].kind)), G, cx.wg, c, cx.lane);
        pw_load(wi, pb_ptr(layers[0].in), pb_of(a.in, pb_sgpr(layers[0].kind)), PW_TIL, G, cx.wg, c, cx.lane);
#pragma nounroll
        for (uint32_t l = 0; l < a.L; l++) {
            asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
            const PbLayer& L = layers[l];
            const uint32_t kind = pb_sgpr(L.kind);
            const PbMat mi = pb_of(a.in, kind), mo = pb_of(a.o, kind);
            if (cx.wg < mi.tiles) {
                __syncthreads();
                __syncthreads();
                if (sh_abort) return;
                v4f acc[PW_TI - PW_TIL];
                pw_mul(wi, mi, c, column(a.W, true), zeros, acc);
#pragma unroll
                for (int t = 0; t < PW_TI - PW_TIL; t++) leave(acc[t], PW_TIL + t, true);
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
                PbSet<PW_TIL, PW_U> wl;
#pragma unroll
                for (int t = 0; t < PW_TIL; t++)
#pragma unroll
                    for (int i = 0; i < PW_U; i++) wl.f[t][i] = *reinterpret_cast<const v8bf*>(slot + (t * PW_U + i) * 1024 + cx.lane * 16);
                v4f acl[PW_TIL];
                pw_mul(wl, mi, c, column(a.W, true), zeros, acl);
#pragma unroll
                for (int t = 0; t < PW_TIL; t++) leave(acl[t], t, true);
                __syncthreads();
            }
            // A head's workgroup: the barriers of what its polling waves do.
            const uint32_t joins = kind == PB_FIRST ? (cx.wg < a.ns.heads ? 3u : 0u) : cx.wg < grouped_roles ? (a.splits > 1 && cx.wg % a.splits == 0 ? 5u : 3u) : 0u;
            const PbLayer& N = layers[min(l + 1, a.L - 1)];
            PbSet<1, PW_U> wo;
            PbSet<PW_TGA, PW_U> wga;
            pw_load(wo, pb_ptr(L.o), mo, 0, G, cx.wg, c, cx.lane);
            pw_load(wga, pb_ptr(L.gate_up), a.gate_up, 0, G, cx.wg, c, cx.lane);
            for (uint32_t j = 0; j < joins; j++) {
                __syncthreads();
                if (sh_abort) return;
            }
            if (!joins) pw_load_lds(slot, pb_ptr(N.in), pb_of(a.in, pb_sgpr(N.kind)), G, cx.wg, c, cx.lane);
            if (on_o) {
                __syncthreads();
                if (sh_abort) return;
                const bool planes = kind == PB_FIRST;
                v4f acc[1];
                pw_mul(wo, mo, c, column(mo.K, planes), zeros, acc);
                leave(acc[0], 0, planes);
                __syncthreads();
            }
            PbSet<PW_TG - PW_TGA, PW_U> wgb;
            if (joins) pw_load_lds(slot, pb_ptr(N.in), pb_of(a.in, pb_sgpr(N.kind)), G, cx.wg, c, cx.lane);
            pw_load(wgb, pb_ptr(L.gate_up), a.gate_up, PW_TGA, G, cx.wg, c, cx.lane);
            if (on_g) {
                __syncthreads();
                __syncthreads();
                if (sh_abort) return;
                const __bf16* xc = column(a.W, true);
                auto some = [&](const auto& w, auto n, int t0) {
#pragma unroll
                    for (int t = 0; t < n.value; t += 2) {
                        PbSet<2, PW_U> two;
#pragma unroll
                        for (int i = 0; i < PW_U; i++) { two.f[0][i] = w.f[t][i]; two.f[1][i] = w.f[t + 1][i]; }
                        v4f acc[2];
                        pw_mul(two, a.gate_up, c, xc, zeros, acc);
                        leave(acc[0], t0 + t, true);
                        leave(acc[1], t0 + t + 1, true);
                    }
                };
                some(wga, std::integral_constant<int, PW_TGA>{}, 0);
                some(wgb, std::integral_constant<int, PW_TG - PW_TGA>{}, PW_TGA);
            }
            if (on_g) __syncthreads();
            PbSet<1, PW_UD> wd;
            pw_load(wd, pb_ptr(L.down), a.down, 0, G, cx.wg, c, cx.lane);
            if (on_o) {
                __syncthreads();
                if (sh_abort) return;
            }
            pw_load(wi, pb_ptr(N.in), pb_of(a.in, pb_sgpr(N.kind)), PW_TIL, G, cx.wg, c, cx.lane);
            if (on_o) {
                v4f acc[1];
                pw_mul(wd, a.down, c, column(a.ff, false), zeros, acc);
                leave(acc[0], 0, false);
                __syncthreads();
            }
        }
    }

    // ---- final norm | output matrix | argmax
    asm volatile("" : "+v"(cx.tid), "+v"(cx.lane));
    stamp(5 * a.L);
    ArgPair best{-INFINITY, 0};
    if (!comp) {
        layer_norm_fetch(a.th, a.tag_base + (a.L - 1) * PB_TAGS + PB_T_DOWN, a.final_norm, false);
        __syncthreads();
        if (sh_abort) return;
    } else {
        PbSet<1, PW_HEAD_U> wh[2];
        const Cur u0{lwv, 0}, u1 = next_of(u0);
        head_load(wh[0], u0);
        head_load(wh[1], u1);
        __syncthreads();
        __syncthreads();
        if (sh_abort) return;
        const __bf16* const x1 = vec + 8 * (cx.lane >> 4);
        v4f acc = (v4f){0.f, 0.f, 0.f, 0.f};
        auto work = [&](const PbSet<1, PW_HEAD_U>& w, Cur u) {
#pragma unroll
            for (int i = 0; i < PW_HEAD_U; i++) {
                const uint32_t k = u.chunk * PW_HEAD_U + i;
                acc = mma16(w.f[0][i], load8(k < mh.K / 32 ? x1 + 32 * k : zeros), acc);
            }
            if (u.chunk + 1 < chunks) return;
            pb_logits(a, u.tile, acc, cx.lane, best);
            acc = (v4f){0.f, 0.f, 0.f, 0.f};
        };
        for (Cur u = u0, v = u1; u.tile < mh.tiles;) {
            work(wh[0], u);
            u = next_of(v);
            head_load(wh[0], u);
            if (v.tile >= mh.tiles) break;
            work(wh[1], v);
            v = next_of(u);
            head_load(wh[1], v);
        }
    }
    pb_choose(a, best, sh_arg, pos, cx);
}

// uk [head][dim][rank] -> [head][rank][dim]
__global__ __launch_bounds__(256) void pb_transpose_kernel(const uint16_t* __restrict__ uk, uint32_t dim, uint32_t rank, uint32_t n, uint16_t* __restrict__ out) {
    const uint32_t i = blockIdx.x * 256 + threadIdx.x;
    if (i >= n) return;
    const uint32_t head = i / (dim * rank), j = i % (dim * rank);
    out[i] = uk[(size_t)head * dim * rank + j % dim * rank + j / dim];
}

// flag <- 1 if one of the weights is larger than PB_LARGEST, infinite or NaN.  Workgroup (.., weights).
constexpr uint32_t PB_LARGEST = 0x4F800000u;
struct PbWeights { const uint32_t* w; uint64_t words; uint32_t f32; };      // bfloat16: two to a word
__global__ __launch_bounds__(256) void pb_large_kernel(const PbWeights* __restrict__ all, uint32_t* flag) {
    const PbWeights m = all[blockIdx.y];
    bool any = false;
    for (uint64_t i = (uint64_t)blockIdx.x * 256 + threadIdx.x; i < m.words; i += (uint64_t)gridDim.x * 256) {
        const uint32_t v = m.w[i];
        any = any || (m.f32 ? (v & 0x7FFFFFFFu) > PB_LARGEST : (v & 0x7FFF0000u) > PB_LARGEST || (v << 16 & 0x7FFF0000u) > PB_LARGEST);
    }
    if (any) *flag = 1;
}

template <typename S> bool pb_same(const S& a, const S& b) { return memcmp(&a, &b, sizeof(S)) == 0; }

// A mixer's input product as far as its rows are read: the raw part and the heads' gates.  (What pads the matrix behind them would make a workgroup that holds nothing else a reader on which
// no later phase depends: it might find its input overwritten, and the step would be given up.)
DenseWeight pb_input(const PbMixer& m) {
    const uint32_t rows = m.kind == MixerKind::LatentAttention ? m.latent.raw_row() + m.latent.heads * m.latent.vdim
                        : m.kind == MixerKind::GroupedAttention ? m.grouped.raw_row() + m.grouped.heads * m.grouped.vdim
                                                                : m.linear.raw_row() + m.linear.heads * m.linear.vdim;
    DenseWeight w = m.in;
    w.N = std::min(w.N, rows);
    return w;
}

}  // namespace

struct PbState {
    PbArgs args{};
    std::vector<void*> owned;
    const void* kernel = nullptr;
    uint32_t grid = 0, lds = 0, n_stamps = 0, heads = 0, window = 0;
    bool cooperative = false, wide = false;
    uint64_t* tagged = nullptr;
    size_t tagged_bytes = 0;
    std::vector<unsigned long long> stamps_host;
    int wall_khz = 0;
    unsigned long long* host_out = nullptr;
    unsigned long long* host_out_dev = nullptr;
    uint32_t seq = 0;
    ~PbState() {
        for (void* p : owned) (void)hipFree(p);
        if (host_out) (void)hipHostFree(host_out);
    }
    template <typename T>
    T* dev(size_t n) {
        void* p = nullptr;
        if (hipMalloc(&p, n < 16 ? 16 : n) != hipSuccess) { (void)hipGetLastError(); return nullptr; }
        owned.push_back(p);
        return static_cast<T*>(p);
    }
};

void pb_destroy(PbState* st) { delete st; }

// Lanes without a key of their own read the last cached row, which an empty cache does not have yet.
bool pb_covers(const PbState* st, int64_t pos) { return st && pos >= 1; }

// Covered: every layer with a feed-forward of one size and activation; latent attention of one shape under elementwise norms with post-norms, or linear and grouped attention, of one
// shape each, under layer norms; what the registers hold.
int32_t pb_create(const PbModelIn& in, PbState** out) {
    *out = nullptr;
    const std::vector<PbLayerIn>& layers = in.layers;
    const bool latent = in.elementwise;
    if (layers.empty() || in.width > (latent ? PB_WIDTH : PW_WIDTH)) return FORGE_HIP_OK;
    const PbLayerIn* of[2] = {nullptr, nullptr};                     // the first layer of each kind
    for (const PbLayerIn& l : layers) {
        const PbMixer& m = *l.mixer;
        const bool grouped = m.kind == MixerKind::GroupedAttention;
        if (latent != (m.kind == MixerKind::LatentAttention) || (latent && !(l.post1.w && l.post2.w))) return FORGE_HIP_OK;
        if (!l.ff || l.ff != layers[0].ff || l.act != layers[0].act) return FORGE_HIP_OK;
        if (!of[grouped]) of[grouped] = &l;
        const PbMixer& f = *of[grouped]->mixer;
        if (m.in.N != f.in.N || m.o.K != f.o.K || !pb_same(m.latent, f.latent) || !pb_same(m.grouped, f.grouped) || !pb_same(m.linear, f.linear)) return FORGE_HIP_OK;
        if (m.kind != MixerKind::LinearAttention && (m.cos_t != f.cos_t || m.sin_t != f.sin_t)) return FORGE_HIP_OK;
    }
    const LatentShape ls = latent ? of[0]->mixer->latent : LatentShape{};
    const LinearShape ns = !latent && of[0] ? of[0]->mixer->linear : LinearShape{};
    const GroupedShape gs = of[1] ? of[1]->mixer->grouped : GroupedShape{};
    if (latent && (ls.q_rank > PB_QR || ls.dim > PB_DIM || ls.cache_row() > PB_ROW || ls.rank > PB_RANK || ls.vdim > PB_VDIM)) return FORGE_HIP_OK;
    if (ns.heads && (ns.dim > 64 || ns.vdim > PB_LVDIM || 64 % (ns.vdim / 4) || ns.rank > PB_LOW || ns.dim * ns.vdim > PB_STATE * 4 * PB_THREADS)) return FORGE_HIP_OK;
    if (gs.heads && (gs.dim > 64 || gs.vdim > 64 || gs.group() > PB_GROUP || !gs.rot_pairs)) return FORGE_HIP_OK;
    if (in.max_seq > 0xFFFFFFFFull / (2 * (uint64_t)std::max({ls.cache_row(), gs.k_row(), gs.v_row(), 1u})) || (uint64_t)in.head.N * in.head.K * 2 > 0xFFFFFFFFull) return FORGE_HIP_OK;

    int dev = 0, coop = 0, cus = 0, khz = 0, per_cu = 0;
    FH_HIP(hipGetDevice(&dev));
    FH_HIP(hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, dev));
    FH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    FH_HIP(hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, dev));
    std::unique_ptr<PbState> st(new PbState());
    st->cooperative = resident_cooperative();
    if (st->cooperative && !coop) return FORGE_HIP_OK;
    PbArgs& a = st->args;
    a.W = in.width; a.Wn = in.ln_n; a.ff = layers[0].ff; a.L = (uint32_t)layers.size();
    a.act = (uint32_t)layers[0].act;
    a.ls = ls; a.gs = gs; a.ns = ns;
    // The fewest workgroups that hold every matrix, then as few tiles each as that many allow.
    uint32_t g = 1;
    auto need = [&](uint32_t N, uint32_t tiles_each) { g = std::max(g, ((N + 15) / 16 + tiles_each - 1) / tiles_each); };
    for (const PbLayerIn* l : of)
        if (l) need(pb_input(*l->mixer).N, PB_TI);
    need(layers[0].gate_up.N, PB_TG);
    need(a.W, 1);
    // ... or, what registers do not hold, all workgroups
    bool& wide = st->wide;
    wide = !latent && (a.W > PB_WIDTH || a.ff > PB_FF || g + std::max({gs.kv_heads, ns.heads, 1u}) > (uint32_t)cus);
    if (wide) g = (uint32_t)cus;
    a.G = g;
    st->heads = latent ? ls.heads : gs.kv_heads;
    if ((wide ? 0u : g) + std::max({st->heads, ns.heads, 1u}) > (uint32_t)cus) return FORGE_HIP_OK;
    if (wide && ns.dim * ns.vdim > (uint32_t)PbLinear<PB_POLL>::STATE * 4 * PB_POLL_THREADS) return FORGE_HIP_OK;
    a.splits_max = st->heads ? std::min(PB_SPLITS, ((uint32_t)cus - (wide ? 0u : g)) / st->heads) : 1u;
    bool fits = true;
    auto mat = [&](const DenseWeight& w, uint32_t tiles_each, uint32_t pieces) {
        const uint32_t rows = wide ? 8 : 16, depth = wide ? 64 : 32;      // of a tile, of a piece (wide: of both halves)
        PbMat m{w.N, w.K, (w.N + rows - 1) / rows, 1, (w.K / depth + PB_COMP - 1) / PB_COMP};
        m.T = (m.tiles + g - 1) / g;
        fits = fits && m.T <= tiles_each && m.per <= pieces && w.K % depth == 0 && w.N % (wide ? 8 : 4) == 0 && (uint64_t)w.N * w.K * 2 <= 0x7FFFFFFFull;
        return m;
    };
    for (int k = 0; k < 2; k++)
        if (of[k]) { a.in[k] = mat(pb_input(*of[k]->mixer), wide ? PW_TI : PB_TI, wide ? PW_U : PB_UI); a.o[k] = mat(of[k]->mixer->o, 1, wide ? PW_U : PB_UO); }
    a.gate_up = mat(layers[0].gate_up, wide ? PW_TG : PB_TG, wide ? PW_U : PB_UI);
    a.down = mat(layers[0].down, 1, wide ? PW_UD : PB_UD);
    if (in.loop.p) a.loop = mat(in.loop, 1, PB_UL);
    a.head = PbMat{in.head.N, in.head.K, (in.head.N + 15) / 16, 1, 1};
    if (!fits || a.in[0].N % 16 || a.in[1].N % 16 || a.gate_up.N % 16) return FORGE_HIP_OK;

    auto up = [](size_t v, size_t m) { return (uint32_t)((v + m - 1) / m * m); };
    a.plane = up(std::max({in.loop.p ? 2 * a.W : a.W, a.ff, a.o[0].K, a.o[1].K}), 32);
    // Planes a quarter of the banks apart (us a token, 135M linear and grouped: 413 -> 410).  Wide: three of the longest vector that comes in planes; longer ones lie over them.
    const uint32_t longest = a.plane;
    a.plane = up(wide ? std::max({a.W, a.o[0].K, a.o[1].K}) : a.plane, 128) + 32;
    a.off_red = wide ? up(std::max(a.plane * 6, longest * 2), 16) : a.plane * 8;
    a.off_stats = a.off_red + (wide ? PW_TG : std::max(PB_TI, PB_TG)) * PB_COMP * 16 * 4;
    a.off_layers = a.off_stats + PB_POLL * 3 * 4;
    a.off_attn = up(a.off_layers + layers.size() * sizeof(PbLayer), 16);
    const size_t attn = latent ? sizeof(PbLatentLds) : wide ? sizeof(PwAttnLds) : sizeof(PbKakiraxLds<PB_WAVES>),
                 recs = latent ? sizeof(PbLatentLds::ct) : wide ? sizeof(PbGroupedLds<PB_POLL>::ct) : sizeof(PbGroupedLds<PB_WAVES>::ct);
    a.off_in = up(a.off_attn + attn, 1024);
    st->lds = wide ? a.off_in + PB_COMP * PW_SLOT : a.off_attn + (uint32_t)attn;
    const uint32_t rec = latent ? ls.rank + 2 : gs.heads ? gs.group() * (gs.vdim + 2) : 0u;
    if (rec) a.splits_max = std::min<uint32_t>(a.splits_max, (uint32_t)(recs / 4 / rec) + 1);
    if (st->lds > PB_LDS) return FORGE_HIP_OK;
    st->window = ls.window;
    st->kernel = wide ? reinterpret_cast<const void*>(decode_block_wide_kernel) : latent ? reinterpret_cast<const void*>(decode_block_kernel<true>) : reinterpret_cast<const void*>(decode_block_kernel<false>);
    FH_HIP(hipFuncSetAttribute(st->kernel, hipFuncAttributeMaxDynamicSharedMemorySize, PB_LDS));
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, st->kernel, PB_THREADS, st->lds) != hipSuccess || per_cu < 1) { (void)hipGetLastError(); return FORGE_HIP_OK; }
    st->grid = (uint32_t)cus;

    std::vector<PbWeights> looked;
    auto look = [&](const void* w, uint64_t n, bool f32) {           // a layer may run with another one's tensors
        if (w && std::none_of(looked.begin(), looked.end(), [&](const PbWeights& l) { return l.w == w; })) looked.push_back(PbWeights{(const uint32_t*)w, f32 ? n : n / 2, f32 ? 1u : 0u});
    };
    auto look_matrix = [&](const DenseWeight& w) { look(w.p, (uint64_t)w.N * w.K, false); };
    look_matrix(in.head);
    look_matrix(in.loop);
    for (const PbLayerIn& l : layers) {
        const PbMixer& m = *l.mixer;
        for (const DenseWeight* w : {&m.in, &m.o, &m.uq, &m.ukv, &l.gate_up, &l.down}) look_matrix(*w);
        for (const float* w : {latent ? l.norm1.w : l.ln1.w, latent ? l.norm2.w : l.ln2.w}) look(w, 2 * (uint64_t)a.W, true);
        const bool lat = m.kind == MixerKind::LatentAttention, lin = m.kind == MixerKind::LinearAttention;
        look(lin ? m.wc : m.wa, lat ? ls.q_rank : lin ? ns.vdim : gs.dim, true);
        if (!lin) look(m.wb, lat ? ls.rank : gs.dim, true);
    }
    PbWeights* looked_dev = st->dev<PbWeights>(looked.size() * sizeof(PbWeights));
    uint32_t *flag = st->dev<uint32_t>(4), large = 0;
    if (!looked_dev || !flag) return FORGE_HIP_OK;
    FH_HIP(hipMemset(flag, 0, 4));
    FH_HIP(hipMemcpy(looked_dev, looked.data(), looked.size() * sizeof(PbWeights), hipMemcpyHostToDevice));
    fh::launch(pb_large_kernel, dim3(128, (uint32_t)looked.size()), 256, 0, nullptr, looked_dev, flag);
    FH_HIP(hipGetLastError());
    FH_HIP(hipMemcpy(&large, flag, 4, hipMemcpyDeviceToHost));
    if (large) return FORGE_HIP_OK;

    std::vector<PbLayer> host(layers.size());
    const uint32_t uk_n = ls.heads * ls.dim * ls.rank;
    std::vector<std::pair<const void*, const __bf16*>> turned;
    for (size_t l = 0; l < layers.size(); l++) {
        const PbLayerIn& i = layers[l];
        const PbMixer& m = *i.mixer;
        PbLayer& h = host[l];
        memset(&h, 0, sizeof(h));
        h.in = (const __bf16*)m.in.p; h.o = (const __bf16*)m.o.p; h.gate_up = (const __bf16*)i.gate_up.p; h.down = (const __bf16*)i.down.p;
        h.kind = m.kind == MixerKind::GroupedAttention ? PB_GROUPED : PB_FIRST;
        h.loop = i.pass_start;
        h.cache = static_cast<uint8_t*>(i.cache);
        h.cache_v = h.cache + m.values_at;
        h.wa = m.wa; h.wb = m.wb; h.wc = m.wc;
        if (!latent) { h.norm1 = i.ln1.w; h.norm2 = i.ln2.w; continue; }
        h.norm1 = i.norm1.w; h.norm2 = i.norm2.w; h.post1 = i.post1.w; h.post2 = i.post2.w;
        h.alpha1 = i.norm1.alpha; h.alpha2 = i.norm2.alpha; h.post_alpha1 = i.post1.alpha; h.post_alpha2 = i.post2.alpha;
        const DynTanh next = l + 1 == layers.size() ? in.final_norm : layers[l + 1].pass_start ? DynTanh{} : layers[l + 1].norm1;
        h.next = next.w; h.next_alpha = next.alpha;
        h.uq = (const __bf16*)m.uq.p;
        h.uv = (const __bf16*)m.ukv.p + uk_n;
        for (const auto& t : turned)
            if (t.first == m.ukv.p) h.uk = t.second;
        if (!h.uk) {
            __bf16* t = st->dev<__bf16>((size_t)uk_n * 2);
            if (!t) return FORGE_HIP_OK;                             // no memory for it: the kernel sequence takes the steps
            fh::launch(pb_transpose_kernel, dim3((uk_n + 255) / 256), 256, 0, nullptr, (const uint16_t*)m.ukv.p, ls.dim, ls.rank, uk_n, (uint16_t*)t);
            turned.emplace_back(m.ukv.p, t);
            h.uk = t;
        }
    }
    PbLayer* dl = st->dev<PbLayer>(host.size() * sizeof(PbLayer));
    const size_t row = a.W, raw = std::max(a.in[0].N, a.in[1].N), outs = std::max(a.o[0].K, a.o[1].K), recs_n = (size_t)st->heads * a.splits_max * rec;
    const size_t n_tagged = 2 * row + raw + outs + a.ff + 2 * (size_t)st->grid + recs_n;
    uint64_t* t = st->dev<uint64_t>(n_tagged * 8);
    if (!dl || !t) return FORGE_HIP_OK;
    FH_HIP(hipMemcpy(dl, host.data(), host.size() * sizeof(PbLayer), hipMemcpyHostToDevice));
    FH_HIP(hipMemset(t, 0, n_tagged * 8));                           // tag 0 is never expected
    st->tagged = t; st->tagged_bytes = n_tagged * 8;
    a.layers = dl;
    a.th = t; t += row;
    a.tl = t; t += row;
    a.traw = t; t += raw;
    a.tout = t; t += outs;
    a.tact = t; t += a.ff;
    a.tpart = t; t += 2 * (size_t)st->grid;
    a.trec = t;
    a.eps = in.ln_eps; a.embed_scale = in.embed_scale; a.cap = in.cap;
    a.table = (const __bf16*)in.table; a.table_ld = in.table_ld; a.table_n = in.table_n;
    a.head_w = (const __bf16*)in.head.p; a.loop_w = (const __bf16*)in.loop.p;
    a.final_norm = in.ln_final;
    const PbLayerIn* rot = latent ? of[0] : of[1];
    if (rot) { a.cos_t = rot->mixer->cos_t; a.sin_t = rot->mixer->sin_t; }
    a.logits = in.logits; a.state = in.state; a.counts = in.counts; a.penalty = 1.0f;
    { const char* e = getenv("FORGE_HIP_PD_TAG_START"); if (e) a.tag_base = (uint32_t)strtoul(e, nullptr, 0); }
    pb_set_poll_limit(st.get(), 0);
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
    st->n_stamps = 5 * a.L + 3;
    *out = st.release();
    return FORGE_HIP_OK;
}

void pb_set_poll_limit(PbState* st, uint32_t n) { st->args.spin_limit = n ? n : 400000u; }
void pb_set_repeat_penalty(PbState* st, float penalty) { st->args.penalty = penalty; }

// As pa_enqueue.
int32_t pb_enqueue(PbState* st, int64_t pos, bool profile, uint32_t token, uint32_t step_seq, hipStream_t s) {
    PbArgs& a = st->args;
    a.token = token;
    a.step_seq = step_seq;
    a.host_out = st->host_out_dev;
    if (a.host_out) a.host_seq = ++st->seq;
    const uint64_t keys = st->window ? std::min<uint64_t>(pos + 1, st->window) : pos + 1;
    // Up to 384 keys one workgroup, which saves the hand-over of parts; from there on four waves a workgroup attend, one to a SIMD, as long as there are workgroups for the keys (1024 keys,
    // us a token: 453 with twelve waves in three parts, 419 with four in eight); then eight, then all, and rounds of those.
    const uint64_t parts = keys <= PB_WAVES * PB_KEYS ? 1 : a.splits_max;
    for (a.attend = 4; !st->wide && a.attend < PB_WAVES && parts * a.attend * PB_KEYS < keys; a.attend += 4) {}
    a.splits = (uint32_t)std::min<uint64_t>(a.splits_max, (keys + a.attend * PB_KEYS - 1) / (a.attend * PB_KEYS));
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
    const hipError_t e = resident_launch(st->kernel, st->grid, PB_THREADS, kargs, st->lds, st->cooperative, s);
    a.stamps = keep;
    if (e != hipSuccess) return fail(FORGE_HIP_ERR_HIP, std::string("resident decode launch: ") + hipGetErrorString(e));
    a.tag_base += PB_TAGS * a.L + 1;
    return FORGE_HIP_OK;
}

// The next token, from the word that the kernel writes last; false: not in use or not in time, wait for the stream instead.
bool pb_wait_token(PbState* st, uint32_t* next) {
    if (!st->host_out || !st->args.host_out) return false;
    const volatile unsigned long long* w = st->host_out;
    const auto t0 = std::chrono::steady_clock::now();
    for (uint32_t spin = 0;; spin++) {
        const unsigned long long v = *w;
        if ((uint32_t)(v >> 32) == st->seq) { *next = (uint32_t)v; return true; }
        if ((spin & 1023u) == 1023u && std::chrono::steady_clock::now() - t0 > std::chrono::milliseconds(200)) return false;
    }
}

// As pa_after_sync.
int32_t pb_after_sync(PbState* st, uint32_t abort_flag, hipStream_t s) {
    if (!abort_flag) return FORGE_HIP_OK;
    PbArgs& a = st->args;
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

// Milliseconds between the phase starts of the last profiled step: five per layer run (input product, attention, output product, gate;up, down), then head and argmax.
int32_t pb_phase_ms(PbState* st, std::vector<float>* out, hipStream_t s) {
    PbArgs& a = st->args;
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
