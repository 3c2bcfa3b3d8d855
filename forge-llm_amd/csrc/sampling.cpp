// The sampler of the generated main.rs (crates/forgellm-codegen-cpu/src/project.rs:505-555), host code: what a caller
// that samples with a temperature runs on the logits `forge_hip_forward` hands back.  Every f32 operation is done in the
// reference's order (sequential sums, one division per element), `exp` is the C library's expf.
//
// What bounds it: passes over the vocabulary on one core.  128 256 logits with top_p 0.9: 9.2 ms with a stable sort of every index
// and a scalar exp, 0.70 ms here -- the order is worked out only down to where top_k or top_p cuts (a radix sort of the candidates), exp
// runs four at a time, and the last two passes visit the entries that are left.  What remains: the order down to the cut and its running
// sum a good half, setting the rest to zero, the maximum and exp 10 % each, the sequential sum of all exponentials 5 %.
#include <math.h>
#include <string.h>

#include <algorithm>

#if !defined(__HIP_DEVICE_COMPILE__) && defined(__x86_64__)
#include <immintrin.h>
#define FH_SAMPLE_AVX2 1
#endif

#include "common.h"
#include "expf_ref.h"

namespace {

uint32_t bits_of(float x) { uint32_t b; memcpy(&b, &x, 4); return b; }

// l[i] = exp(l[i] - shift)
void exp_scalar(float* l, uint64_t n, float shift) {
    for (uint64_t i = 0; i < n; i++) l[i] = fh::expf_ref<true>(l[i] - shift);
}
#ifdef FH_SAMPLE_AVX2
// The same operations in the same order, four at a time (fused multiply-adds round once in either form).
__attribute__((target("avx2,fma"))) void exp_avx2(float* l, uint64_t n, float shift) {
    alignas(32) static const struct Table {
        uint64_t t[32];
        Table() { for (int i = 0; i < 32; i++) t[i] = fh::expf_detail::tab(i); }
    } table;
    namespace ex = fh::expf_detail;
    const __m256d inv = _mm256_set1_pd(ex::InvLn2N), round = _mm256_set1_pd(ex::Shift), one = _mm256_set1_pd(1.0);
    const __m256d c0 = _mm256_set1_pd(ex::C0), c1 = _mm256_set1_pd(ex::C1), c2 = _mm256_set1_pd(ex::C2);
    const __m256i low5 = _mm256_set1_epi64x(31);
    const __m128 sh = _mm_set1_ps(shift), least = _mm_set1_ps(ex::Least), most = _mm_set1_ps(ex::Most), inf = _mm_set1_ps(INFINITY);
    uint64_t i = 0;
    for (; i + 4 <= n; i += 4) {
        const __m128 x = _mm_sub_ps(_mm_loadu_ps(l + i), sh);
        __m256d z = _mm256_mul_pd(inv, _mm256_cvtps_pd(x));
        __m256d kd = _mm256_add_pd(z, round);
        const __m256i ki = _mm256_castpd_si256(kd);
        kd = _mm256_sub_pd(kd, round);
        const __m256d r = _mm256_sub_pd(z, kd);
        __m256i t = _mm256_i64gather_epi64((const long long*)table.t, _mm256_and_si256(ki, low5), 8);
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
    exp_scalar(l + i, n - i, shift);
}
#endif
void exp_all(float* l, uint64_t n, float shift) {
#ifdef FH_SAMPLE_AVX2
    static const bool wide = __builtin_cpu_supports("avx2") && __builtin_cpu_supports("fma");
    if (wide) { exp_avx2(l, n, shift); return; }
#endif
    exp_scalar(l, n, shift);
}

// The entries of l (none negative, none NaN) from the largest down, lower index first among equals, as far as someone asks.
// Numbers that are not negative are ordered like their bits: a histogram of the upper 16 says how far down a batch of at least `want`
// more entries reaches, and the batch is sorted by all 32.
struct Descending {
    struct Entry { uint32_t bits, index; };
    static constexpr uint32_t BUCKETS = 0x8000;
    const float* l;
    uint64_t n;
    std::vector<uint32_t> count;
    std::vector<Entry> order, spare;      // the sorted prefix, and room to sort in
    uint32_t floor = BUCKETS;             // buckets from here up are in `order`
    // Few entries, of which a first batch of `want` would take most, are sorted at once: the histogram alone takes 15 to 25 us (50 entries with
    // top_p 3.5 us against 29, 1000 with top_p 45 against 69, 300 with top_k 40 11 against 21; but 1000 with top_k 40 take 26 with it).
    Descending(const float* l_, uint64_t n_, uint64_t want) : l(l_), n(n_) {
        if (n <= want || n <= 384) {
            order.resize(n);
            for (uint64_t i = 0; i < n; i++) order[i] = {bits_of(l[i]) & 0x7FFFFFFFu, (uint32_t)i};
            sort_from(0);
            floor = 0;
            return;
        }
        count.assign(BUCKETS, 0u);
        for (uint64_t i = 0; i < n; i++) count[(bits_of(l[i]) >> 16) & (BUCKETS - 1)]++;      // (-0.0 is a zero like the other)
    }
    // The passes over all entries stand alone: inside their callers they lose registers and alignment to the exceptional paths around them
    // (128256 entries with top_p 0.9 415 us there, 372 here; 32000 with top_k 40 102 and 91).
    __attribute__((noinline)) static void collect(const float* l, uint64_t n, uint32_t floor, uint32_t above, Entry* to) {
        for (uint64_t i = 0; i < n; i++) {
            const uint32_t b = bits_of(l[i]) & 0x7FFFFFFFu, k = b >> 16;
            if (k >= floor && k < above) *to++ = {b, (uint32_t)i};
        }
    }
    // Sets what does not stay to 0 and lists what does.
    __attribute__((noinline)) static void cut(float* l, uint64_t n, const uint8_t* stays, uint32_t* kept) {
        for (uint64_t i = 0; i < n; i++) {
            if (stays[i]) *kept++ = (uint32_t)i;
            else l[i] = 0.0f;
        }
    }
    void sort_from(size_t at) {
        std::stable_sort(order.begin() + at, order.end(), [](const Entry& a, const Entry& b) { return a.bits > b.bits; });
    }
    // Appends a batch; false: everything is there already.
    bool extend(uint64_t want) {
        if (floor == 0) return false;
        const uint32_t above = floor;
        uint64_t m = 0;
        while (floor > 0 && m < want) m += count[--floor];
        const size_t at = order.size();
        order.resize(at + m);
        collect(l, n, floor, above, order.data() + at);
        // they came in index order: any stable sort by bits will do
        if (m < 4096) { sort_from(at); return true; }
        spare.resize(m);
        Entry *from = order.data() + at, *to = spare.data();
        for (int shift = 0; shift < 33; shift += 11) {
            uint32_t place[2048] = {};
            for (uint64_t i = 0; i < m; i++) place[(from[i].bits >> shift) & 2047u]++;
            uint32_t sum = 0;
            for (int b = 2047; b >= 0; b--) { const uint32_t c = place[b]; place[b] = sum; sum += c; }
            for (uint64_t i = 0; i < m; i++) to[place[(from[i].bits >> shift) & 2047u]++] = from[i];
            std::swap(from, to);
        }
        memcpy(order.data() + at, from, m * sizeof(Entry));      // three passes: the result sits in `spare`
        return true;
    }
};

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
    for (uint64_t i = 0; i < n; i++) FH_CHECK(l[i] == l[i], "sample: a logit is NaN");
    if (temperature <= 0.0f) {
        uint64_t best = 0;
        for (uint64_t i = 1; i < n; i++) if (l[i] >= l[best]) best = i;        // max_by keeps the last maximum
        *out = (uint32_t)best;
        return FORGE_HIP_OK;
    }
    for (uint64_t i = 0; i < n; i++) l[i] /= temperature;
    float max_val = -INFINITY;
    for (uint64_t i = 0; i < n; i++) max_val = l[i] > max_val ? l[i] : max_val;
    exp_all(l, n, max_val);                                 // f32::exp = the C library's expf
    float sum = 0.0f;
    for (uint64_t i = 0; i < n; i++) sum += l[i];
    bool nan = false;
    for (uint64_t i = 0; i < n; i++) { l[i] /= sum; nan |= l[i] != l[i]; }
    FH_CHECK(!nan, "sample: a probability is NaN");
    const bool cut_k = top_k > 0 && top_k < n, cut_p = top_p > 0.0f && top_p < 1.0f;
    std::vector<uint32_t> kept;                             // entries that are not set to 0, ascending; used when `few`
    bool few = false;
    if (cut_k || cut_p) {
        // Largest first, equal ones by index: what lies past the first top_k goes, and what follows once the sum so far (which takes every
        // entry, zeros included, and never falls) exceeds top_p -- the entry that crosses the threshold too (project.rs:535-540).
        try {
            uint64_t batch = cut_k ? std::min<uint64_t>(top_k, 4096) : 1024;
            Descending d(l, n, batch);
            const uint64_t most = cut_k ? top_k : n;
            uint64_t keep = 0;
            float cumsum = 0.0f;
            bool crossed = false;
            while (!crossed && keep < most) {
                if (keep == d.order.size()) {
                    if (!d.extend(batch)) break;
                    batch *= 4;
                    continue;
                }
                if (cut_p) {
                    cumsum += l[d.order[keep].index];
                    if (cumsum > top_p) { crossed = true; break; }
                }
                keep++;
            }
            // (no crossing and no top_k: everything stays)
            if (crossed || keep < n) {
                few = true;
                kept.resize(keep);
                std::vector<uint8_t> stays(n, 0);
                for (uint64_t k = 0; k < keep; k++) stays[d.order[k].index] = 1;
                Descending::cut(l, n, stays.data(), kept.data());
            }
        } catch (const std::bad_alloc&) {
            return fh::fail(FORGE_HIP_ERR_INVALID, "sample: out of memory");
        }
    }
    // Zeros neither change a sum nor a quotient: where entries were cut, only those that are left are visited.
    const uint64_t left = few ? kept.size() : n;
    auto at = [&](uint64_t k) -> uint64_t { return few ? kept[k] : k; };
    sum = 0.0f;
    for (uint64_t k = 0; k < left; k++) sum += l[at(k)];
    if (sum > 0.0f)
        for (uint64_t k = 0; k < left; k++) l[at(k)] /= sum;
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
        cumsum += l[at(k)];
        if (cumsum >= r) { *out = (uint32_t)at(k); break; }
    }
    return FORGE_HIP_OK;
}

}  // extern "C"
