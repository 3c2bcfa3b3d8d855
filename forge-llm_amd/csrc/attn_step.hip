// Attention of one query over an fp16 KV cache for a caller's own loop (attention_flash, attention_sliding: emit.rs:598-715), flat or paged.  (A model's step has the
// kernels of attn_decode.hip, whose sums the resident kernel repeats bit for bit.)
//
// What bounds it: launches and latency; a cache of a few hundred rows is a microsecond's worth of memory traffic, 8192 of 8 KV heads 3.4 us at the rate of a large copy.  So
//   * a short context is done by one workgroup per KV head, in one launch;
//   * a longer one is cut into parts, as many as are resident at once.  Each of the workgroup's eight waves requests its 32 keys and values together, a round of them, and
//     all of it is on its way before the query is looked at; parts meet in attn_step_combine_kernel;
//   * scores and weighted values are products on the matrix unit.  On the vector unit they were 250 instructions for 8 keys of 4 heads, 3 us of a part of 256.
// The query and the weights stay 32-bit: the 16 columns of a product hold four query heads, each as three fp16 planes that add up to it (x = hi + lo + rest, to 2^-33 of
// the largest element of a head, to 2^-36 of the largest weight), whose results are added in 32-bit.
// us from a caller's loop, the pair of attn_decode.hip / this: 32 heads on 8 of 64, 17..257 rows 10.5 / 7.9, 512 10.8 / 9.7, 4096 11.0 / 10.6, 8192 13.4 / 11.6, 32768
// 26.9 / 19.5; 48 on 16, 8192 rows 16.3 / 13.1; 128 on 32, 512 rows 15.2 / 9.9, 8192 27.4 / 18.8.  Distance from 64 bits, the pair / this: 1.32 / 1.27e-7 at 33 rows, 1.80 / 1.64 at
// 1024, 2.08 / 1.95 at 8192 (24 random caches each).
#include <algorithm>

#include "attn_decode_math.h"
#include "common.h"
#include "dense.h"
#include "device_utils.h"
#include "lds_transpose.h"

namespace fh {

namespace {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

constexpr int AS_WAVES = 8;
constexpr uint32_t AS_KEYS = 32, AS_STRIDE = AS_KEYS + 8;      // keys of a wave's round; LDS row of transposed values and of weights
constexpr float AS_WEIGHT = 4096.f;                            // weights go into their planes times this: the third one's last bit is 2^-36

// Plane 0, 1 or 2 of x; 3: nothing.
__device__ __forceinline__ _Float16 as_plane(float x, uint32_t plane) {
    const _Float16 hi = (_Float16)x;
    const float r = x - (float)hi;
    const _Float16 lo = (_Float16)r, rest = (_Float16)(r - (float)lo);
    return plane == 0 ? hi : plane == 1 ? lo : plane == 2 ? rest : (_Float16)0.0f;
}
// Sum over the planes, in all of their lanes.
__device__ __forceinline__ float as_sum(float v) { return lane_xor_add<8>(lane_xor_add<4>(v)); }

// A wave's sums by single keys: lane d (and d + 64) has the columns.  rec: [GT][HD sums, maximum, weight sum].
template <int HD, int GT, typename Row>
__device__ __forceinline__ void as_one_by_one(const float* q, const uint16_t* kc, const uint16_t* vc, float* rec, Row row_of, uint32_t h0, uint32_t kvh, uint32_t kv_stride, uint32_t first0,
                                           uint32_t step, uint32_t t1, uint32_t lane) {
    const float scale = 1.0f / sqrtf((float)HD);
    for (uint32_t g = 0; g < GT; g++) {
        float m = -INFINITY, l = 0.f, a[2] = {0.f, 0.f};
        for (uint32_t first = first0; first < t1; first += step)
            for (uint32_t t = first; t < min(t1, first + AS_KEYS); t++) {
                const size_t at = row_of(t) * kv_stride + kvh * HD;
                float d = 0.f;
                for (uint32_t c = lane; c < HD; c += 64) d = fmaf(q[(size_t)(h0 + g) * HD + c], f16_bits_to_f32(kc[at + c]), d);
                d = wave_sum(d) * scale;
                // a score of -inf has the weight 0, also ahead of all others (0 times an infinite value is no number); fmaxf passes NaN over, the weight does not
                const float m_new = fmaxf(m, d), alpha = m == -INFINITY ? 0.f : __expf(m - m_new), p = d == -INFINITY ? 0.f : __expf(d - m_new);
                m = m_new;
                l = fmaf(l, alpha, p);
                for (uint32_t c = lane, i = 0; c < HD; c += 64, i++) a[i] = fmaf(p, f16_bits_to_f32(vc[at + c]), a[i] * alpha);
            }
        for (uint32_t c = lane, i = 0; c < HD; c += 64, i++) rec[g * (HD + 2) + c] = a[i];
        if (lane == 0) { rec[g * (HD + 2) + HD] = m; rec[g * (HD + 2) + HD + 1] = l; }
    }
}

// Workgroup (query heads h0 .. + GT of one KV head, part).  `direct`, one part: the result; else records [head][part][HD sums, maximum, weight sum].
template <int HD, int GT, bool PAGED>
__global__ __launch_bounds__(AS_WAVES * 64) void attn_step_kernel(const float* __restrict__ q, const uint16_t* __restrict__ kc, const uint16_t* __restrict__ vc, float* __restrict__ out,
                                                                  uint32_t seq, uint32_t kv_heads, uint32_t gsize, uint32_t start, uint32_t chunk, uint32_t direct, PageTable pt) {
    constexpr int P = HD / 32;                   // pieces of 32 columns
    constexpr int REC = HD + 2;
    constexpr uint32_t STRIP = (HD + 16) * AS_STRIDE;
    static_assert(STRIP * 2 >= GT * REC * 4, "a wave's strip holds its sums");
    __shared__ __align__(16) _Float16 lds[AS_WAVES * STRIP];
    __shared__ uint32_t pt_s[PAGED ? PAGE_ENTRIES_MAX : 1];
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), l16 = lane & 15u, lg = lane >> 4;
    const uint32_t gpk = gsize / GT, kvh = blockIdx.x / gpk, h0 = kvh * gsize + blockIdx.x % gpk * GT, split = blockIdx.y;
    const uint32_t t0 = min(seq, start + split * chunk), t1 = min(seq, t0 + chunk), kv_stride = kv_heads * HD;
    const uint32_t head = min(l16 & 3u, (uint32_t)GT - 1), plane = (l16 & 3u) < GT ? l16 >> 2 : 3u;      // this lane's column
    _Float16* ct = lds + wave * STRIP;           // [HD][AS_STRIDE]: values, transposed
    _Float16* pw = ct + HD * AS_STRIDE;          // [16][AS_STRIDE]: weights, a row per column

    const uint32_t pt_first = PAGED ? t0 >> pt.shift : 0, n_entries = PAGED && t1 > t0 ? ((t1 - 1) >> pt.shift) - pt_first + 1 : 0;
    const bool pt_near = n_entries <= PAGE_ENTRIES_MAX;      // a part's table entries in LDS, where they fit
    if (PAGED && pt_near) {
        for (uint32_t i = tid; i < n_entries; i += AS_WAVES * 64) pt_s[i] = pt.table[pt_first + i];
        __syncthreads();
    }
    auto row_of = [&](uint32_t t) -> size_t {
        if (!PAGED) return t;
        const uint32_t at = t >> pt.shift;
        return ((size_t)(pt_near ? pt_s[at - pt_first] : pt.table[at]) << pt.shift) + (t & ((1u << pt.shift) - 1));
    };
    struct Keys { uint4 k[2][P], v[2][P]; };
    auto load = [&](Keys& r, uint32_t first) {
#pragma unroll
        for (int t = 0; t < 2; t++) {
            const size_t at = row_of(min(first + 16 * t + l16, t1 - 1)) * kv_stride + kvh * HD + 8 * lg;      // rows past the part: its last one
#pragma unroll
            for (int s = 0; s < P; s++) r.k[t][s] = __builtin_bit_cast(uint4, *reinterpret_cast<const Half8*>(kc + at + 32 * s));
#pragma unroll
            for (int s = 0; s < P; s++) r.v[t][s] = __builtin_bit_cast(uint4, *reinterpret_cast<const Half8*>(vc + at + 32 * s));
        }
    };
    float m = -INFINITY, l = 0.f;
    v4f o[2 * P];
#pragma unroll
    for (int i = 0; i < 2 * P; i++) o[i] = (v4f){0.f, 0.f, 0.f, 0.f};
    const uint32_t first0 = t0 + wave * AS_KEYS, step = AS_WAVES * AS_KEYS;
    Keys now, next;
    if (first0 < t1) load(now, first0);
    // The query's column, times a power of two that brings its largest element to 2^13 .. 2^14.
    v8h qf[P];
    float unscale;
    {
        float x[P][8], mx = 0.f;
        const float* row = q + (size_t)(h0 + head) * HD + 8 * lg;
#pragma unroll
        for (int s = 0; s < P; s++)
#pragma unroll
            for (int j = 0; j < 8; j++) { x[s][j] = row[32 * s + j]; mx = fmaxf(mx, fabsf(x[s][j])); }
        mx = lane_xor_max<32>(lane_xor_max<16>(mx));
        const int e = mx > 0.f && mx < INFINITY ? 14 - __builtin_amdgcn_frexp_expf(mx) : 0;
        unscale = ldexpf(1.0f / sqrtf((float)HD), -e);
#pragma unroll
        for (int s = 0; s < P; s++)
#pragma unroll
            for (int j = 0; j < 8; j++) qf[s][j] = as_plane(ldexpf(x[s][j], e), plane);
    }
    const v4f zero = (v4f){0.f, 0.f, 0.f, 0.f};
    auto attend = [&](const Keys& r, uint32_t first) {
        v4f s[2];
        float mx = -INFINITY;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            // pieces and rounds are added on the vector unit, which rounds to nearest
            s[t] = zero;
#pragma unroll
            for (int i = 0; i < P; i++) s[t] += __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(v8h, r.k[t][i]), qf[i], zero, 0, 0, 0);
            // a key that is not there has no value either (0 * v is not 0 for an infinite v)
            const bool there = first + 16 * t + l16 < t1;
#pragma unroll
            for (int i = 0; i < P; i++) {
                uint4 v = r.v[t][i];
                if (!there) v = make_uint4(0u, 0u, 0u, 0u);
                lay_down_transposed<__bf16, AS_STRIDE>(reinterpret_cast<__bf16*>(ct), __builtin_bit_cast(v8bf, v), 32 * i, 16 * t, l16, lg);
            }
            // register r: key first + 16 t + 4 lg + r of this column's head
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float d = as_sum(s[t][k]) * unscale;
                s[t][k] = first + 16 * t + 4 * lg + k < t1 ? d : -INFINITY;
                mx = fmaxf(mx, s[t][k]);
            }
        }
        const float m_new = fmaxf(m, lane_xor_max<32>(lane_xor_max<16>(mx)));
        // no score above -inf so far: weights of 0
        const float alpha = m == -INFINITY ? 0.f : expf(m - m_new);
        m = m_new;
        l *= alpha;
#pragma unroll
        for (int t = 0; t < 2; t++) {
            v4h w;
#pragma unroll
            for (int k = 0; k < 4; k++) {
                const float p = s[t][k] == -INFINITY ? 0.f : expf(s[t][k] - m_new);
                l += p;
                w[k] = as_plane(p * AS_WEIGHT, plane);
            }
            *reinterpret_cast<v4h*>(pw + l16 * AS_STRIDE + 16 * t + 4 * lg) = w;
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");      // LDS operations of one wave execute in order
        __builtin_amdgcn_wave_barrier();
        const v8h w = *reinterpret_cast<const v8h*>(pw + l16 * AS_STRIDE + 8 * lg);
#pragma unroll
        for (int i = 0; i < 2 * P; i++) {
            const v4f sum = __builtin_amdgcn_mfma_f32_16x16x32_f16(*reinterpret_cast<const v8h*>(ct + (16 * i + l16) * AS_STRIDE + 8 * lg), w, zero, 0, 0, 0);
#pragma unroll
            for (int k = 0; k < 4; k++) o[i][k] = fmaf(o[i][k], alpha, sum[k]);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    for (uint32_t first = first0; first < t1; first += step) {
        const bool more = first + step < t1;
        if (more) load(next, first + step);
        attend(now, first);
        if (more) now = next;
    }
    // An infinity times a plane of 0 is no number: a wave that meets one does its keys once more, a head and a key at a time, in 32-bit throughout.
    float bad = l;
#pragma unroll
    for (int i = 0; i < 2 * P; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) bad = fmaf(o[i][k], 0.f, bad);
    if (__any(!(bad < INFINITY))) {
        as_one_by_one<HD, GT>(q, kc, vc, reinterpret_cast<float*>(ct), row_of, h0, kvh, kv_stride, first0, step, t1, lane);
    } else {
    // the wave's sums where its strip was, then the workgroup's
    l = lane_xor_add<32>(lane_xor_add<16>(l));
    float* rec = reinterpret_cast<float*>(ct);
#pragma unroll
    for (int i = 0; i < 2 * P; i++)
#pragma unroll
        for (int k = 0; k < 4; k++) o[i][k] = as_sum(o[i][k]) * (1.0f / AS_WEIGHT);
    if (l16 < GT) {
#pragma unroll
        for (int i = 0; i < 2 * P; i++)
#pragma unroll
            for (int k = 0; k < 4; k++) rec[l16 * REC + 16 * i + 4 * lg + k] = o[i][k];
        if (lg == 0) { rec[l16 * REC + HD] = m; rec[l16 * REC + HD + 1] = l; }
    }
    }
    __syncthreads();
    for (uint32_t e = tid; e < GT * HD; e += AS_WAVES * 64) {
        const uint32_t g = e / HD, d = e % HD;
        float ms[AS_WAVES], ls[AS_WAVES], os[AS_WAVES], mm = -INFINITY;
#pragma unroll
        for (int w = 0; w < AS_WAVES; w++) {
            const float* r = reinterpret_cast<const float*>(lds + w * STRIP) + g * REC;
            ms[w] = r[HD]; ls[w] = r[HD + 1]; os[w] = r[d];
            mm = fmaxf(mm, ms[w]);
        }
#pragma unroll
        for (int w = 0; w < AS_WAVES; w++) {
            const float x = ms[w] == -INFINITY ? 0.f : expf(ms[w] - mm);
            os[w] *= x;
            ls[w] *= x;
        }
        // the waves in pairs: a third of the rounding of a sum in a row
#pragma unroll
        for (int n = AS_WAVES / 2; n; n /= 2)
#pragma unroll
            for (int w = 0; w < n; w++) { os[w] += os[w + n]; ls[w] += ls[w + n]; }
        if (direct) {
            out[(size_t)(h0 + g) * HD + d] = os[0] * (1.0f / ls[0]);
        } else {
            float* to = out + ((size_t)(h0 + g) * gridDim.y + split) * REC;
            to[d] = os[0];
            if (d == 0) { to[HD] = mm; to[HD + 1] = ls[0]; }
        }
    }
}

// Workgroup = head, thread = column: the parts' records together, in pairs as above (sums over 32 parts in a row were the larger share of a long context's error).
template <int HD>
__global__ __launch_bounds__(HD) void attn_step_combine_kernel(const float* __restrict__ rec, uint32_t nsplit, float* __restrict__ out) {
    constexpr int REC = HD + 2;
    __shared__ float weight_s[DECODE_SPLITS], total_s;
    const uint32_t d = threadIdx.x;
    const float* base = rec + (size_t)blockIdx.x * nsplit * REC;
    float part[DECODE_SPLITS];
#pragma unroll
    for (uint32_t i = 0; i < DECODE_SPLITS; i++) part[i] = base[min(i, nsplit - 1) * REC + d];      // all on their way
    if (d < 64) {
        const float m = d < nsplit ? base[d * REC + HD] : -INFINITY, mm = wave_max(m), w = m == -INFINITY ? 0.f : expf(m - mm);
        const float total = wave_sum(d < nsplit ? w * base[d * REC + HD + 1] : 0.f);
        if (d < DECODE_SPLITS) weight_s[d] = w;
        if (d == 0) total_s = total;
    }
    __syncthreads();
#pragma unroll
    for (uint32_t i = 0; i < DECODE_SPLITS; i++) part[i] = i < nsplit ? weight_s[i] * part[i] : 0.f;
#pragma unroll
    for (uint32_t n = DECODE_SPLITS / 2; n; n /= 2)
#pragma unroll
        for (uint32_t i = 0; i < n; i++) part[i] += part[i + n];
    out[(size_t)blockIdx.x * HD + d] = part[0] * (1.0f / total_s);
}

// What this kernel takes; the pair, which reads rows of any width by the lane, takes the rest.
// One workgroup per KV head, us, the pair / one: heads of 64, 512 rows 10.8 / 9.7, 1000 equal to parts; of 96 (32 on 32), 129 rows 10.3 / 7.9, 257 10.2 / 9.3, 500 slower;
// of 128 (24 on 8), 100 rows 10.5 / 9.0, 257 equal, 500 slower (a wave's round is 128 bytes a lane there and its registers hold no second one).
// Parts, heads of 64 by three or four to a workgroup: above.  Two or one leave most columns of a product empty: 32 on 32, 8192 rows, 17.3 / 18.6; 14 on 2 12.0 / 12.9.  Longer rows: 32 on
// 32 of 96, 8192 rows, 26.8 / 39.
// A part is 128 rows or what makes 256 workgroups: 140 registers a lane let one be on a CU, and a second turn of them costs more than longer parts (64 on 8, 3000 rows: 14.5 us
// with 24 parts, 11.2 with 16, the pair 13.4).
constexpr uint32_t as_one(uint32_t hd) { return hd == 64 ? 512 : hd == 96 ? 256 : 128; }
constexpr uint32_t AS_PART = 128, AS_CUS = 256;

// Query heads that share a workgroup.
uint32_t as_heads(uint32_t gsize) { return gsize % 4 == 0 ? 4 : gsize % 3 == 0 ? 3 : gsize % 2 == 0 ? 2 : 1; }

// Parts of the context: 1 if one workgroup a KV head does it, 0 if the pair does.
uint32_t as_parts(uint32_t keys, uint32_t hd, uint32_t heads, uint32_t gsize) {
    if (keys <= as_one(hd)) return 1;
    const uint32_t gt = as_heads(gsize), full = std::min(DECODE_SPLITS, AS_CUS / (heads / gt));
    return hd == 64 && gt >= 3 && full ? std::min(full, (keys + AS_PART - 1) / AS_PART) : 0;
}

template <int HD, int GT>
void launch_heads(const float* q, const uint16_t* kc, const uint16_t* vc, float* out, uint32_t seq, uint32_t start, uint32_t parts, bool apart, uint32_t heads, uint32_t kv_heads,
                  float* ws, const PageTable& pt, hipStream_t s) {
    const uint32_t gsize = heads / kv_heads, keys = seq - start;
    const uint32_t chunk = ((keys + parts - 1) / parts + AS_KEYS - 1) / AS_KEYS * AS_KEYS, nsplit = (keys + chunk - 1) / chunk;      // no part is empty
    const dim3 grid(kv_heads * (gsize / GT), nsplit);
    const uint32_t direct = nsplit == 1 && apart;
    float* to = direct ? out : ws;
    if (pt.table) fh::launch(attn_step_kernel<HD, GT, true>, grid, AS_WAVES * 64, 0, s, q, kc, vc, to, seq, kv_heads, gsize, start, chunk, direct, pt);
    else fh::launch(attn_step_kernel<HD, GT, false>, grid, AS_WAVES * 64, 0, s, q, kc, vc, to, seq, kv_heads, gsize, start, chunk, direct, pt);
    if (!direct) fh::launch(attn_step_combine_kernel<HD>, heads, HD, 0, s, ws, nsplit, out);
}

template <int HD>
void launch_hd(const float* q, const uint16_t* kc, const uint16_t* vc, float* out, uint32_t seq, uint32_t start, uint32_t parts, bool apart, uint32_t heads, uint32_t kv_heads,
               float* ws, const PageTable& pt, hipStream_t s) {
    switch (as_heads(heads / kv_heads)) {
        case 4: launch_heads<HD, 4>(q, kc, vc, out, seq, start, parts, apart, heads, kv_heads, ws, pt, s); break;
        case 3: launch_heads<HD, 3>(q, kc, vc, out, seq, start, parts, apart, heads, kv_heads, ws, pt, s); break;
        case 2: launch_heads<HD, 2>(q, kc, vc, out, seq, start, parts, apart, heads, kv_heads, ws, pt, s); break;
        default: launch_heads<HD, 1>(q, kc, vc, out, seq, start, parts, apart, heads, kv_heads, ws, pt, s);
    }
}

}  // namespace

void launch_attn_step(const float* q, const uint16_t* kc, const uint16_t* vc, float* out, uint32_t seq, uint32_t heads, uint32_t kv_heads, uint32_t hd, uint32_t window, void* workspace,
                      hipStream_t s, PageTable pt) {
    const uint32_t start = window != 0 && seq > window ? seq - window : 0u, keys = seq - start, parts = as_parts(keys, hd, heads, heads / kv_heads);
    float* ws = reinterpret_cast<float*>(workspace);
    // One launch stores results while other workgroups read: only with a result apart from all that is read, or in place of the query (a workgroup stores its own heads).  Where a
    // table's pages lie is not known here.
    const size_t result = (size_t)heads * hd * 4, cache = (size_t)seq * kv_heads * hd * 2;
    const bool apart = !pt.table && (out == q || !overlap(out, result, q, result)) && !overlap(out, result, kc, cache) && !overlap(out, result, vc, cache);
    if (!parts) launch_attn_decode(q, kc, vc, out, nullptr, nullptr, seq, nullptr, heads, kv_heads, hd, window, workspace, s, pt);
    else if (hd == 64) launch_hd<64>(q, kc, vc, out, seq, start, parts, apart, heads, kv_heads, ws, pt, s);
    else if (hd == 96) launch_hd<96>(q, kc, vc, out, seq, start, parts, apart, heads, kv_heads, ws, pt, s);
    else launch_hd<128>(q, kc, vc, out, seq, start, parts, apart, heads, kv_heads, ws, pt, s);
}

}  // namespace fh
