// The sampler of the generated main.rs (crates/forgellm-codegen-cpu/src/project.rs:505-555), host code: what a caller
// that samples with a temperature runs on the logits `forge_hip_forward` hands back.  Every f32 operation is done in the
// reference's order (sequential sums, one division per element), `exp` is the C library's expf.
//
// What bounds it: one chain of 32-bit additions over the whole vocabulary, whose order is part of the result.  Everything else is arranged
// around it: exp and a histogram of the results run beside the chain, the histogram says above which number the entries are that top_k or
// top_p can reach, those alone are divided, sorted (their values; who they are matters only at the cut) and summed up, and the rest is
// cleared.  128 256 logits with top_p 0.9 (one in nine stays): 0.23 ms, of which the chain with all beside it 0.15; 0.75 ms with passes of their own for each step and an order worked
// out in batches of four times the size, 9.2 ms with a stable sort of every index and a scalar exp.
#include <math.h>
#include <string.h>

#include <algorithm>

#if !defined(__HIP_DEVICE_COMPILE__) && defined(__x86_64__)
#include <immintrin.h>
#define FH_SAMPLE_X86 1
#endif

#include "common.h"
#include "expf_ref.h"

namespace {

uint32_t bits_of(float x) { uint32_t b; memcpy(&b, &x, 4); return b; }
float float_of(uint32_t b) { float x; memcpy(&x, &b, 4); return x; }

// l[i] = exp(l[i] / temperature - shift)
void exp_scalar(float* l, uint64_t n, float temperature, float shift) {
    for (uint64_t i = 0; i < n; i++) l[i] = fh::expf_ref<true>(l[i] / temperature - shift);
}
#ifdef FH_SAMPLE_X86
alignas(64) static const struct ExpTable {
    uint64_t t[32];
    ExpTable() { for (int i = 0; i < 32; i++) t[i] = fh::expf_detail::tab(i); }
} exp_table;
// The same operations in the same order, four or eight at a time (fused multiply-adds round once in either form).
__attribute__((target("avx2,fma"))) void exp_avx2(float* l, uint64_t n, float temperature, float shift) {
    namespace ex = fh::expf_detail;
    const __m256d inv = _mm256_set1_pd(ex::InvLn2N), round = _mm256_set1_pd(ex::Shift), one = _mm256_set1_pd(1.0);
    const __m256d c0 = _mm256_set1_pd(ex::C0), c1 = _mm256_set1_pd(ex::C1), c2 = _mm256_set1_pd(ex::C2);
    const __m256i low5 = _mm256_set1_epi64x(31);
    const __m128 by = _mm_set1_ps(temperature), sh = _mm_set1_ps(shift), least = _mm_set1_ps(ex::Least), most = _mm_set1_ps(ex::Most), inf = _mm_set1_ps(INFINITY);
    uint64_t i = 0;
    for (; i + 4 <= n; i += 4) {
        const __m128 x = _mm_sub_ps(_mm_div_ps(_mm_loadu_ps(l + i), by), sh);
        __m256d z = _mm256_mul_pd(inv, _mm256_cvtps_pd(x));
        __m256d kd = _mm256_add_pd(z, round);
        const __m256i ki = _mm256_castpd_si256(kd);
        kd = _mm256_sub_pd(kd, round);
        const __m256d r = _mm256_sub_pd(z, kd);
        __m256i t = _mm256_i64gather_epi64((const long long*)exp_table.t, _mm256_and_si256(ki, low5), 8);
        t = _mm256_add_epi64(t, _mm256_slli_epi64(ki, 47));
        z = _mm256_fmadd_pd(c0, r, c1);
        const __m256d r2 = _mm256_mul_pd(r, r);
        __m256d y = _mm256_fmadd_pd(c2, r, one);
        y = _mm256_fmadd_pd(z, r2, y);
        __m128 f = _mm256_cvtpd_ps(_mm256_mul_pd(y, _mm256_castsi256_pd(t)));
        f = _mm_blendv_ps(f, _mm_setzero_ps(), _mm_cmplt_ps(x, least));
        f = _mm_blendv_ps(f, inf, _mm_cmpgt_ps(x, most));
        f = _mm_blendv_ps(f, _mm_add_ps(x, x), _mm_cmpunord_ps(x, x));
        _mm_storeu_ps(l + i, f);
    }
    exp_scalar(l + i, n - i, temperature, shift);
}
#define FH_AVX512 __attribute__((target("avx512f,avx512vl,avx512dq,avx512bw,avx2,fma")))
FH_AVX512 void exp_avx512(float* l, uint64_t n, float temperature, float shift) {
    namespace ex = fh::expf_detail;
    const __m512d inv = _mm512_set1_pd(ex::InvLn2N), round = _mm512_set1_pd(ex::Shift), one = _mm512_set1_pd(1.0);
    const __m512d c0 = _mm512_set1_pd(ex::C0), c1 = _mm512_set1_pd(ex::C1), c2 = _mm512_set1_pd(ex::C2);
    const __m512i t0 = _mm512_load_si512(exp_table.t), t1 = _mm512_load_si512(exp_table.t + 8), t2 = _mm512_load_si512(exp_table.t + 16), t3 = _mm512_load_si512(exp_table.t + 24);
    const __m512i bit4 = _mm512_set1_epi64(16);
    const __m256 by = _mm256_set1_ps(temperature), sh = _mm256_set1_ps(shift), least = _mm256_set1_ps(ex::Least), most = _mm256_set1_ps(ex::Most);
    uint64_t i = 0;
    for (; i + 8 <= n; i += 8) {
        const __m256 x = _mm256_sub_ps(_mm256_div_ps(_mm256_loadu_ps(l + i), by), sh);
        __m512d z = _mm512_mul_pd(inv, _mm512_cvtps_pd(x));
        __m512d kd = _mm512_add_pd(z, round);
        const __m512i ki = _mm512_castpd_si512(kd);
        kd = _mm512_sub_pd(kd, round);
        const __m512d r = _mm512_sub_pd(z, kd);
        __m512i t = _mm512_mask_blend_epi64(_mm512_test_epi64_mask(ki, bit4), _mm512_permutex2var_epi64(t0, ki, t1), _mm512_permutex2var_epi64(t2, ki, t3));
        t = _mm512_add_epi64(t, _mm512_slli_epi64(ki, 47));
        z = _mm512_fmadd_pd(c0, r, c1);
        const __m512d r2 = _mm512_mul_pd(r, r);
        __m512d y = _mm512_fmadd_pd(c2, r, one);
        y = _mm512_fmadd_pd(z, r2, y);
        __m256 f = _mm512_cvtpd_ps(_mm512_mul_pd(y, _mm512_castsi512_pd(t)));
        f = _mm256_mask_blend_ps(_mm256_cmp_ps_mask(x, least, _CMP_LT_OQ), f, _mm256_setzero_ps());
        f = _mm256_mask_blend_ps(_mm256_cmp_ps_mask(x, most, _CMP_GT_OQ), f, _mm256_set1_ps(INFINITY));
        f = _mm256_mask_blend_ps(_mm256_cmp_ps_mask(x, x, _CMP_UNORD_Q), f, _mm256_add_ps(x, x));
        _mm256_storeu_ps(l + i, f);
    }
    exp_scalar(l + i, n - i, temperature, shift);
}
#endif

// The entries of l whose bits are `floor` or more, in order: their bits to `bits`, their places to `index` (room for 16 more than there are).
uint64_t collect_scalar(const float* l, uint64_t from, uint64_t n, uint32_t floor, uint32_t* bits, uint32_t* index) {
    uint64_t m = 0;
    for (uint64_t i = from; i < n; i++) {
        bits[m] = bits_of(l[i]);
        index[m] = (uint32_t)i;
        m += bits_of(l[i]) >= floor;
    }
    return m;
}
#ifdef FH_SAMPLE_X86
FH_AVX512 uint64_t collect_avx512(const float* l, uint64_t from, uint64_t n, uint32_t floor, uint32_t* bits, uint32_t* index) {
    const __m512i least = _mm512_set1_epi32((int)floor), step = _mm512_set1_epi32(16);
    __m512i at = _mm512_add_epi32(_mm512_set1_epi32((int)from), _mm512_set_epi32(15, 14, 13, 12, 11, 10, 9, 8, 7, 6, 5, 4, 3, 2, 1, 0));
    uint64_t m = 0, i = from;
    for (; i + 16 <= n; i += 16, at = _mm512_add_epi32(at, step)) {
        const __m512i v = _mm512_loadu_si512(l + i);
        const __mmask16 in = _mm512_cmpge_epu32_mask(v, least);
        _mm512_storeu_si512(bits + m, _mm512_maskz_compress_epi32(in, v));
        _mm512_storeu_si512(index + m, _mm512_maskz_compress_epi32(in, at));
        m += (uint64_t)__builtin_popcount(in);
    }
    return m + collect_scalar(l, i, n, floor, bits + m, index + m);
}
#endif

struct Forms {
    void (*exp)(float*, uint64_t, float, float) = exp_scalar;
    uint64_t (*collect)(const float*, uint64_t, uint64_t, uint32_t, uint32_t*, uint32_t*) = collect_scalar;
    Forms() {
#ifdef FH_SAMPLE_X86
        if (__builtin_cpu_supports("avx2") && __builtin_cpu_supports("fma")) exp = exp_avx2;
        if (__builtin_cpu_supports("avx512f") && __builtin_cpu_supports("avx512vl") && __builtin_cpu_supports("avx512dq") && __builtin_cpu_supports("avx512bw") &&
            __builtin_cpu_supports("fma")) {
            exp = exp_avx512;
            collect = collect_avx512;
        }
#endif
    }
};
const Forms& forms() {
    static const Forms f;
    return f;
}

// Numbers that are not negative are ordered like their bits.  The histogram of the exponentials (0 .. 1) goes by the upper 13: sixteen buckets
// to a power of two.
constexpr int BUCKET_SHIFT = 19;
constexpr uint32_t BUCKETS = (0x3F800000u >> BUCKET_SHIFT) + 1;

// l = exp(l / temperature - max), the sum of all in order, and (COUNT) their histogram.  In blocks: one block's exponentials run beside the
// additions of the one before.
template <bool COUNT>
float exp_and_sum(float* l, uint64_t n, float temperature, float max_val, uint32_t* count) {
    const auto exp = forms().exp;
    float sum = 0.0f;
    for (uint64_t b = 0; b < n; b += 32) {
        const uint64_t e = std::min(n, b + 32);
        exp(l + b, e - b, temperature, max_val);
        for (uint64_t i = b; i < e; i++) {
            sum += l[i];
            if (COUNT) count[std::min(bits_of(l[i]) >> BUCKET_SHIFT, BUCKETS - 1)]++;
        }
    }
    return sum;
}

// Ascending.  m entries, room for as many in `spare`; none above `most`.
void sort_keys(uint32_t* keys, uint32_t* spare, uint64_t m, uint32_t most) {
    if (m < 512) { std::sort(keys, keys + m); return; }
    const int width = most ? 32 - __builtin_clz(most) : 1, passes = (width + 10) / 11, bits = (width + passes - 1) / passes;
    uint32_t place[3][2048] = {};
    const uint32_t mask = (1u << bits) - 1;
    for (uint64_t i = 0; i < m; i++)
        for (int p = 0; p < passes; p++) place[p][(keys[i] >> (p * bits)) & mask]++;
    uint32_t *from = keys, *to = spare;
    for (int p = 0; p < passes; p++) {
        uint32_t sum = 0;
        for (uint32_t b = 0; b <= mask; b++) { const uint32_t c = place[p][b]; place[p][b] = sum; sum += c; }
        for (uint64_t i = 0; i < m; i++) to[place[p][(from[i] >> (p * bits)) & mask]++] = from[i];
        std::swap(from, to);
    }
    if (from != keys) memcpy(keys, from, m * 4);
}

// What top_k and top_p leave of l (exponentials): probabilities (l / sum) and places, in order.
struct Kept {
    bool all = false;                       // everything stays
    std::vector<uint32_t> index;
    std::vector<float> p;
};
// Largest first, equal ones by index: what lies past the first `most` goes, and what follows once the sum so far (which takes every entry, zeros
// included, and never falls) exceeds top_p -- the entry that crosses the threshold too (project.rs:535-540).
void cut(const float* l, uint64_t n, float sum, const uint32_t* count, uint64_t most, bool cut_p, float top_p, Kept* out) {
    std::vector<uint32_t> room;
    auto middle = [&](uint32_t b) { return (double)count[b] * float_of((b << BUCKET_SHIFT) | (1u << (BUCKET_SHIFT - 1))); };      // of a bucket's numbers, off by 1/33 at most
    // Little is left out: what the buckets hold from the top says too little about it, being off by as much when one entry has most of the sum; what the others hold does.  (Nothing of
    // note lies below the first that is looked at.)  By the former alone all entries were sorted as soon as one had most of the sum: 128 256 of a spread of 8, top_p 0.99, 1.95 ms, this way 0.34.
    const bool by_rest = cut_p && top_p > 0.96f;
    const double out_of = (1.0 - (double)top_p) * sum;
    double others = 0.0;
    if (by_rest)
        for (uint32_t b = bits_of((float)(out_of / (1024.0 * n))) >> BUCKET_SHIFT; b < BUCKETS; b++)
            if (count[b]) others += middle(b);
    // Buckets from the top until they hold `most` entries, or a little more than top_p of the sum; where that turns out to be too few, a little more than that, and in the end all.
    const double more[3] = {1.0 + 1.0 / 512, 1.0 + 1.0 / 32, INFINITY}, less[3] = {15.0 / 16, 1.0 / 4, -INFINITY};
    for (int attempt = 0;; attempt++) {
        uint32_t floor = BUCKETS;
        uint64_t m = 0;
        double mass = 0.0, rest = others;
        const double enough = cut_p ? (double)top_p * sum * more[attempt] : INFINITY, few = out_of * less[attempt];
        while (floor > 0 && m < most && (by_rest ? rest > few : mass < enough)) {
            floor--;
            m += count[floor];
            if (count[floor]) {
                mass += middle(floor);
                rest -= middle(floor);
            }
        }
        // The order is that of the quotients, and numbers that differ may have the same: what has the quotient of the least number of the last
        // bucket stands beside it, whichever bucket it is in (a bit pattern or two below; many where quotients are denormal).
        uint32_t least = floor << BUCKET_SHIFT;
        if (least > 0) {
            const float p = float_of(least) / sum;
            uint32_t below = 0;                                    // float_of(below - 1) / sum < p <= float_of(least) / sum
            while (below < least) {
                const uint32_t mid = below + (least - below) / 2;
                if (float_of(mid) / sum < p) below = mid + 1;
                else least = mid;
            }
            for (uint32_t b = least >> BUCKET_SHIFT; b < floor; b++) m += count[b];      // room for as many
        }
        room.resize(3 * (m + 16));
        uint32_t *key = room.data(), *index = key + m + 16, *spare = index + m + 16;
        m = forms().collect(l, 0, n, least, key, index);
        std::vector<uint32_t> sorted(m);
        for (uint64_t i = 0; i < m; i++) key[i] = bits_of(float_of(key[i]) / sum);
        uint32_t hi = 0, lo = UINT32_MAX;
        for (uint64_t i = 0; i < m; i++) { hi = std::max(hi, key[i]); lo = std::min(lo, key[i]); }
        for (uint64_t i = 0; i < m; i++) sorted[i] = hi - key[i];
        sort_keys(sorted.data(), spare, m, m ? hi - lo : 0);
        const uint64_t end = std::min(m, most);
        uint64_t keep = 0;
        bool crossed = false;
        if (cut_p) {
            float cumsum = 0.0f;
            for (; keep < end; keep++) {
                cumsum += float_of(hi - sorted[keep]);
                if (cumsum > top_p) { crossed = true; break; }
            }
        } else keep = end;
        if (!crossed && keep < most && least > 0) {
            if (m > n / 2) attempt = 1;      // most of them anyway: all
            continue;
        }
        if (!crossed && keep == n) { out->all = true; return; }
        out->index.resize(keep + 1);
        out->p.resize(keep + 1);
        if (keep == 0) { out->index.clear(); out->p.clear(); return; }
        // equal to the last that stays: as many as it takes, lower index first
        const uint32_t last = hi - sorted[keep - 1];
        uint64_t equal = 0, at = 0;
        while (equal < keep && hi - sorted[keep - 1 - equal] == last) equal++;
        for (uint64_t i = 0; i < m && at < keep; i++) {
            out->index[at] = index[i];
            out->p[at] = float_of(key[i]);
            const bool ties = key[i] == last && equal > 0;
            if (ties) equal--;
            at += key[i] > last || ties;
        }
        out->index.resize(keep);
        out->p.resize(keep);
        return;
    }
}

}  // namespace

extern "C" {

// apply_repeat_penalty, project.rs:505-513: once per entry of `recent`, in order.
int32_t forge_hip_apply_repeat_penalty(float* logits_host, uint64_t n, const uint32_t* recent_host, uint64_t n_recent, float penalty) {
    FH_CHECK(logits_host && (recent_host || n_recent == 0), "apply_repeat_penalty: null pointer");
    if (penalty <= 1.0f) return FORGE_HIP_OK;
    for (uint64_t k = 0; k < n_recent; k++) {
        const uint64_t idx = recent_host[k];
        if (idx < n) {
            if (logits_host[idx] > 0.0f) logits_host[idx] /= penalty;
            else logits_host[idx] *= penalty;
        }
    }
    return FORGE_HIP_OK;
}

// sample, project.rs:515-555.  `logits_host` is overwritten like the reference's `&mut [f32]` (it ends up holding the
// final probabilities).  temperature <= 0 returns the last maximum (argmax, project.rs:501-503) and leaves the
// state alone.  A NaN makes the reference panic (`partial_cmp().unwrap()`): FORGE_HIP_ERR_INVALID here.
// Equal probabilities: the reference sorts with `sort_unstable_by`, whose order among equal keys is unspecified;
// here the lower index comes first.
int32_t forge_hip_sample(float* logits_host, uint64_t n, float temperature, uint64_t top_k, float top_p, uint64_t* rng_state,
                         uint32_t* out) {
    FH_CHECK(logits_host && rng_state && out, "sample: null pointer");
    FH_CHECK(n >= 1 && n <= 0xFFFFFFFFull, "sample: the number of logits must be in 1 .. 2^32-1");
    float* l = logits_host;
    // the largest, by signed integers of the same order; a NaN's are the largest without their sign
    int32_t top = INT32_MIN;
    uint32_t size = 0;
    for (uint64_t i = 0; i < n; i++) {
        const int32_t b = (int32_t)bits_of(l[i]);
        top = std::max(top, b ^ ((b >> 31) & 0x7FFFFFFF));
        size = std::max(size, (uint32_t)b & 0x7FFFFFFFu);
    }
    FH_CHECK(size <= 0x7F800000u, "sample: a logit is NaN");
    if (temperature <= 0.0f) {
        uint64_t best = 0;
        for (uint64_t i = 1; i < n; i++) if (l[i] >= l[best]) best = i;        // max_by keeps the last maximum
        *out = (uint32_t)best;
        return FORGE_HIP_OK;
    }
    // (division by a positive number keeps the order, so the largest quotient is the largest logit's; f32::exp = the C library's expf)
    const float max_val = float_of((uint32_t)(top ^ ((top >> 31) & 0x7FFFFFFF))) / temperature;
    const bool cut_k = top_k > 0 && top_k < n, cut_p = top_p > 0.0f && top_p < 1.0f;
    Kept kept;                                              // of the entries that are not set to 0
    kept.all = !cut_k && !cut_p;
    float sum;
    if (kept.all) {
        sum = exp_and_sum<false>(l, n, temperature, max_val, nullptr);
        FH_CHECK(sum == sum, "sample: a probability is NaN");           // some exponential is 1, none above: only a NaN makes a quotient NaN
    } else {
        uint32_t count[BUCKETS] = {};
        sum = exp_and_sum<true>(l, n, temperature, max_val, count);
        FH_CHECK(sum == sum, "sample: a probability is NaN");
        try {
            cut(l, n, sum, count, cut_k ? top_k : n, cut_p, top_p, &kept);
        } catch (const std::bad_alloc&) {
            return fh::fail(FORGE_HIP_ERR_INVALID, "sample: out of memory");
        }
    }
    // Zeros neither change a sum nor a quotient: where entries were cut, only those that are left are visited.
    float* p = kept.all ? l : kept.p.data();
    const uint64_t left = kept.all ? n : kept.p.size();
    auto at = [&](uint64_t k) -> uint64_t { return kept.all ? k : kept.index[k]; };
    if (kept.all) for (uint64_t i = 0; i < n; i++) l[i] /= sum;
    float total = 0.0f;
    for (uint64_t k = 0; k < left; k++) total += p[k];
    if (total > 0.0f)
        for (uint64_t k = 0; k < left; k++) p[k] /= total;
    if (!kept.all) {
        memset(l, 0, n * sizeof(float));
        for (uint64_t k = 0; k < left; k++) l[kept.index[k]] = p[k];
    }
    uint64_t s = *rng_state;                                  // xorshift64, project.rs:545-547
    s ^= s << 13;
    s ^= s >> 7;
    s ^= s << 17;
    *rng_state = s;
    const float r = (float)s / (float)UINT64_MAX;
    *out = (uint32_t)(n - 1);
    if (r <= 0.0f) { *out = 0; return FORGE_HIP_OK; }         // the first entry's sum reaches it, whatever the entry
    float cumsum = 0.0f;
    for (uint64_t k = 0; k < left; k++) {
        cumsum += p[k];
        if (cumsum >= r) { *out = (uint32_t)at(k); break; }
    }
    return FORGE_HIP_OK;
}

}  // extern "C"
