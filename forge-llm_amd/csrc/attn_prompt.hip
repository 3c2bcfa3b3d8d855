// Attention of a prompt's rows in bfloat16 or 32-bit: keys and values per head (or per group of heads), an optional key part that all
// heads share, an optional window, a gate on the output.  T: __bf16 or float (dense.h); scores, softmax and sums are 32-bit in both.
#include <hip/hip_runtime.h>

#include "common.h"
#include "dense.h"
#include "device_utils.h"

namespace fh {

constexpr float LOG2E = 1.4426950408889634f;

// Workgroup = 8 waves: 8 / KG groups of 32 consecutive queries of one head, each shared by KG waves that take 32 keys each of every tile
// of 32 KG and merge their (maximum, sum, output) at the end, which cuts the longest chain of dependent tile steps to a KG-th.  Both products are
// computed transposed (S^T = K Q^T, O^T = V^T P^T): a lane owns one query, so the softmax statistics are per-lane scalars, and the exponentiated
// scores are already the second product's operand.  Scores stay in the base-2 domain.
//   bfloat16  Tiles go straight into one of two pairs of LDS buffers while the other is worked, one barrier a step, 32 columns (64 bytes) of 16 rows at a time,
//             so that a load is all of K's own part, or of the shared part, or of V.  V is transposed on its way out of LDS (ds_read_b64_tr_b16).
//   32-bit    Through registers into one buffer (K row-major: the head's own part, the shared part; V transposed), two barriers a step.
// What bounds it: up to a few hundred workgroups the chain of steps, each a trip through LDS, two products and the exponentials between them; then the VALU (exponentials,
// maxima, conversions) beside the matrix unit.  In bfloat16 a step through registers took 1.8 us, half of it the loads' issue and the writes to LDS, and its registers left
// one workgroup to a compute unit; now 1.1, and two.  us, before / now: 9 heads of 64 + 32 with a window of 1024, 902 tokens 18.4 / 15.2, 2502 36.0 / 23.3, 4000 47.1 /
// 29.7; 32/8 heads of 64 902 23.2 / 16.0, 2502 92.7 / 54.0; 24/8 of 128 2502 101.9 / 90.1; 16 of 128 + 64 902 40.1 / 33.0, 4000 169 / 147; 33 tokens the same.
// DQ >= dim + rot and DV >= vdim: the register tiles' sizes; columns past the real ones are zero.
constexpr uint32_t LP_THREADS = 512;
constexpr uint32_t LP_RSRC_FLAGS = 0x00020000;   // raw buffer, 32-bit data format
template <typename T, int DQ> constexpr bool prompt_four() { return sizeof(T) == 2 && DQ <= 96; }      // four waves to a SIMD
template <typename T, int DQ, int DV, int KG> constexpr uint32_t prompt_lds() {
    const uint32_t tiles = sizeof(T) == 2 ? 2 * 32 * KG * (DQ + DV) * 2 : (32 * KG * (DQ + 16 / sizeof(T)) + DV * (32 * KG + 8 / sizeof(T))) * sizeof(T),
                   merge = 8 / KG * (KG - 1) * 64 * 18 * 4;
    return tiles > merge ? tiles : merge;
}

#define FH_LDS3(p) ((__attribute__((address_space(3))) void*)(p))

// V fragments of 32 keys x 32 N columns: f[j][d] = keys 16 j + 4 lh .. + 3 and + 8 of column 32 d + lane % 32, from rows of 64 bytes, CHUNK bytes from one 32
// columns to the next; at0, at1: LDS addresses of this lane's part of the first keys and of those 8 further on.  Its own waits: ahead of a transposing read of its
// own the compiler waits for everything that is on its way into LDS, that is for the next tiles in the middle of a step.
#define FH_TR(dst, at, off) "ds_read_b64_tr_b16 " dst ", " at " offset:" off "\n"
template <int N, int CHUNK>
__device__ __forceinline__ void read_v(v8bf (&f)[2][N], uint32_t at0, uint32_t at1) {
    v4bf r[4 * N];
    if constexpr (N == 1)
        asm volatile(FH_TR("%0", "%4", "0") FH_TR("%1", "%5", "0") FH_TR("%2", "%4", "1024") FH_TR("%3", "%5", "1024") "s_waitcnt lgkmcnt(0)"
                     : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]) : "v"(at0), "v"(at1));
    else
        asm volatile(FH_TR("%0", "%8", "0") FH_TR("%1", "%9", "0") FH_TR("%2", "%8", "1024") FH_TR("%3", "%9", "1024")
                     FH_TR("%4", "%8", "%10") FH_TR("%5", "%9", "%10") FH_TR("%6", "%8", "%10+1024") FH_TR("%7", "%9", "%10+1024") "s_waitcnt lgkmcnt(0)"
                     : "=&v"(r[0]), "=&v"(r[1]), "=&v"(r[2]), "=&v"(r[3]), "=&v"(r[4]), "=&v"(r[5]), "=&v"(r[6]), "=&v"(r[7])
                     : "v"(at0), "v"(at1), "n"(CHUNK));
#pragma unroll
    for (int d = 0; d < N; d++)
#pragma unroll
        for (int j = 0; j < 2; j++) f[j][d] = __builtin_shufflevector(r[4 * d + 2 * j], r[4 * d + 2 * j + 1], 0, 1, 2, 3, 4, 5, 6, 7);
}
#undef FH_TR

// Chunks [C0, C1) of a tile, each 16 RG rows of 32 columns, into LDS: load j (a wave's are wave, wave + 8, ...) fills 1 KB with 16 rows; lane -> 16-byte piece.  Columns
// [0, n) come from `a`, those from there to `all` from `b`, columns past that and rows past the last read 0.  Piece c of row r lies at c ^ (r / 4 % 4) of its 64 bytes:
// sixteen rows at one piece (fragments of K) touch all banks, and four rows (V) do as they are.
template <uint32_t RG, uint32_t C0, uint32_t C1, typename T>
__device__ __forceinline__ void direct_rows(const T* a, uint32_t a_row, uint32_t n, const T* b, uint32_t b_row, uint32_t all, uint32_t rows, uint32_t a_lane, uint32_t b_lane,
                                            uint8_t* lds, uint32_t wave) {
#pragma unroll
    for (uint32_t j0 = C0 * RG / 8 * 8; j0 < C1 * RG; j0 += 8) {
        const uint32_t j = j0 + wave;
        if ((j0 < C0 * RG && j < C0 * RG) || (j0 + 8 > C1 * RG && j >= C1 * RG)) continue;
        const uint32_t col = (j / RG - C0) * 32, r = j % RG * 16;
        const bool of_a = col < n;
        const uint32_t st = of_a ? a_row : b_row, at_lane = of_a ? a_lane : b_lane;
        const uint64_t from = (uint64_t)((of_a ? a + col : b + (col - n)) + r * st);
        const uint32_t records = r < rows && col < all ? (min(rows - r, 16u) - 1) * st * 2 + 64 : 0u;
        // (readfirstlane: all of it is uniform, and a descriptor word in a vector register would cost a loop over its values around the load)
        const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)from), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(from >> 32));
        const __amdgpu_buffer_rsrc_t rsrc =
            __builtin_amdgcn_make_buffer_rsrc((void*)(((uint64_t)hi << 32) | lo), 0, (uint32_t)__builtin_amdgcn_readfirstlane((int)records), LP_RSRC_FLAGS);
        __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, FH_LDS3(lds + j * 1024), 16, at_lane, 0, 0, 0);
    }
}

template <typename T, int DQ, int DV, int KG>
__global__ __launch_bounds__(LP_THREADS) __attribute__((amdgpu_waves_per_eu(prompt_four<T, DQ>() ? 4 : 2)))
void attn_prompt_kernel(PromptAttn sh, const T* __restrict__ q, const T* __restrict__ kbuf, const T* __restrict__ vbuf, const T* __restrict__ shared,
                        const T* __restrict__ gate, T* __restrict__ out, uint32_t M, uint32_t base_pos) {
    typedef typename Vec<T>::x4 x4;
    typedef typename Vec<T>::x8 x8;
    constexpr uint32_t KT = 32 * KG, QB = 32 * (8 / KG), NT = LP_THREADS, PAD = 16 / sizeof(T);
    constexpr uint32_t KS = DQ + PAD, VS = KT + 8 / sizeof(T);         // LDS row strides
    constexpr uint32_t NS = DQ / 16, ND = DV / 32;
    constexpr uint32_t KTOTAL = KT * DQ / 8, VTOTAL = (KT / 2) * (DV / 4);       // pieces of a tile
    constexpr uint32_t KP = (KTOTAL + NT - 1) / NT, VP = (VTOTAL + NT - 1) / NT;
    constexpr bool DIRECT = sizeof(T) == 2, FOUR = prompt_four<T, DQ>();
    constexpr uint32_t CHUNK = KT * 64, NCK = DQ / 32, NC = NCK + DV / 32, PAIR = NC * CHUNK;      // DIRECT: 32 columns of a tile, such chunks of K, of K and V, their bytes
    extern __shared__ __attribute__((aligned(16))) uint8_t ap_lds[];
    T* Ks = reinterpret_cast<T*>(ap_lds);
    T* Vt = Ks + KT * KS;

    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6)), lq = lane & 31, lh = lane >> 5;
    const uint32_t qg = wave / KG, kh = wave % KG;       // query group, 32 keys of every key tile
    // latest (longest) query tiles first
    const uint32_t head = blockIdx.x % sh.heads, ntq = gridDim.x / sh.heads;
    const uint32_t q0 = (ntq - 1 - blockIdx.x / sh.heads) * QB;
    const uint32_t kvh = head / sh.group, kv_lo = sh.kv_lo, ld_out = sh.ld_out;
    const uint32_t dq = sh.dim + sh.rot, window = sh.window ? sh.window : 0xFFFFFFFFu;
    // A folder may give any scale.  32-bit: scores are scaled, then masked.  bfloat16: they are masked and compared ahead of their scale, which wants it above 0: a negative one
    // turns the query's sign, and where it is less than the least normal number (or 0) that number stands in, by which the weights of all finite products are alike.
    const bool turned = DIRECT && sh.scale < 0.f;
    const float c2 = DIRECT ? fmaxf(fabsf(sh.scale * LOG2E), 0x1p-126f) : sh.scale * LOG2E, later = DIRECT ? c2 : 1.f;
    const uint32_t qrow = q0 + qg * 32 + lq, qpos = base_pos + qrow;

    // requested at once: a row past the last takes the last one's, columns past dq any of the row's
    x8 qf[NS];
    auto load_q = [&]() {
        const T* row = q + ((size_t)min(qrow, M - 1) * sh.heads + head) * dq;
#pragma unroll
        for (uint32_t s = 0; s < NS; s++) qf[s] = load8(row + (16 * s < dq ? 16 * s : 0u) + 8 * lh);
#pragma unroll
        for (uint32_t s = 0; s < NS; s++)
            if (16 * s >= dq) qf[s] = zero8<T>();
        if (turned) {
#pragma unroll
            for (uint32_t s = 0; s < NS; s++) qf[s] = -qf[s];
        }
    };
    v16f oacc[ND];
#pragma unroll
    for (uint32_t d = 0; d < ND; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) oacc[d][r] = 0.f;
    float m_run = -INFINITY, l_run = 0.f;

    const uint32_t total = base_pos + M;
    const uint32_t wg_max = base_pos + min(q0 + QB, M) - 1, wg_min = base_pos + q0;
    const bool wave_active = q0 + qg * 32 < M;
    const uint32_t wave_min = wg_min + qg * 32, wave_max = base_pos + min(q0 + qg * 32 + 32, M) - 1;
    auto first_visible = [&](uint32_t p) { return p >= window ? p - window + 1 : 0u; };
    const uint32_t wave_lo = first_visible(wave_min), last_lo = first_visible(wave_max);
    // tiles are counted from kv_lo, the first row that is there
    const uint32_t tile0 = (first_visible(wg_min) - kv_lo) / KT, ntiles = (wg_max - kv_lo) / KT + 1;

    const uint32_t kst = sh.k_row, vst = sh.v_row, cst = sh.shared_row;
    x8 kreg[KP];
    x4 va[VP], vb[VP];
    auto load_tile = [&](uint32_t kt) {
#pragma unroll
        for (uint32_t i = 0; i < KP; i++) {
            const uint32_t idx = tid + NT * i, key = idx / (DQ / 8), d = idx % (DQ / 8) * 8, t = kv_lo + kt * KT + key;
            if (idx >= KTOTAL || t >= total || d >= dq) kreg[i] = zero8<T>();
            else kreg[i] = d < sh.dim ? load8(kbuf + (size_t)(t - kv_lo) * kst + kvh * sh.dim + d)
                                      : load8(shared + (size_t)t * cst + (d - sh.dim));
        }
#pragma unroll
        for (uint32_t i = 0; i < VP; i++) {
            const uint32_t idx = tid + NT * i, kp = idx / (DV / 4), d = idx % (DV / 4) * 4, t = kv_lo + kt * KT + 2 * kp;
            const T* src = vbuf + (size_t)(t - kv_lo) * vst + kvh * sh.vdim + d;
            const bool in = idx < VTOTAL && d < sh.vdim;
            x4 z;
#pragma unroll
            for (int e = 0; e < 4; e++) z[e] = (T)0.f;
            va[i] = in && t < total ? *reinterpret_cast<const x4*>(src) : z;
            vb[i] = in && t + 1 < total ? *reinterpret_cast<const x4*>(src + vst) : z;
        }
    };
    auto store_tile = [&]() {
#pragma unroll
        for (uint32_t i = 0; i < KP; i++) {
            const uint32_t idx = tid + NT * i, key = idx / (DQ / 8), d = idx % (DQ / 8) * 8;
            if (idx < KTOTAL) store8(Ks + key * KS + d, kreg[i]);
        }
        // the two keys' values of one column side by side
#pragma unroll
        for (uint32_t i = 0; i < VP; i++) {
            const uint32_t idx = tid + NT * i, kp = idx / (DV / 4), d = idx % (DV / 4) * 4;
            if (idx >= VTOTAL) continue;
#pragma unroll
            for (int e = 0; e < 4; e++) {
                struct __attribute__((aligned(2 * sizeof(T)))) Pair { T a, b; } p = {va[i][e], vb[i][e]};
                *reinterpret_cast<Pair*>(Vt + (d + e) * VS + 2 * kp) = p;
            }
        }
    };

    const uint32_t l_row = lane >> 2, l_col = ((lane & 3) ^ ((lane >> 4) & 3)) * 16;
    const uint32_t k_lane = l_row * kst * 2 + l_col, c_lane = l_row * cst * 2 + l_col, v_lane = l_row * vst * 2 + l_col;
    auto direct_tile = [&](uint32_t kt, uint32_t buf) {
        const uint32_t r0 = kt * KT;
        direct_rows<KT / 16, 0, NCK>(kbuf + (size_t)r0 * kst + kvh * sh.dim, kst, sh.dim, shared + (size_t)(kv_lo + r0) * cst, cst, dq, total - kv_lo - r0, k_lane, c_lane,
                                     ap_lds + buf * PAIR, wave);
        direct_rows<KT / 16, NCK, NC>(vbuf + (size_t)r0 * vst + kvh * sh.vdim, vst, sh.vdim, vbuf, 0, sh.vdim, total - kv_lo - r0, v_lane, 0, ap_lds + buf * PAIR, wave);
    };
    const uint32_t k_at = (kh * 32 + lq) * 64 + ((lh ^ ((lq >> 2) & 3)) * 16);       // odd steps of 16 columns: ^ 32
    const uint32_t v_row = 4 * lh + ((lane & 15) >> 2), v_piece = 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1);
    const uint32_t v_at = NCK * CHUNK + (kh * 32 + v_row) * 64 + ((v_piece ^ lh) * 16) + (lane & 1) * 8;      // 8 keys further on: + 512, ^ 32

    if constexpr (DIRECT) direct_tile(tile0, tile0 & 1);
    else load_tile(tile0);
    load_q();
    for (uint32_t kt = tile0; kt < ntiles; kt++) {
        const uint8_t* pair = ap_lds + (kt & 1) * PAIR;
        if constexpr (DIRECT) {
            __builtin_amdgcn_s_waitcnt(0);        // this wave's share of the step's tiles is in LDS,
            __syncthreads();                      // and so is everyone's; nobody reads the other pair any more
            if (kt + 1 < ntiles) direct_tile(kt + 1, (kt + 1) & 1);
        } else {
            __syncthreads();                      // the previous tile has been read
            store_tile();
            __syncthreads();
            if (kt + 1 < ntiles) load_tile(kt + 1);
        }
        const uint32_t k0 = kv_lo + kt * KT + kh * 32;                                     // the wave's 32 keys
        if (!(wave_active && k0 <= wave_max && k0 + 32 > wave_lo)) continue;       // all in the wave's future, or before its windows
        auto k_frag = [&](uint32_t s) {
            if constexpr (DIRECT) return *reinterpret_cast<const x8*>(pair + (k_at ^ ((s & 1) * 32)) + (s >> 1) * CHUNK);
            else return load8(Ks + (kh * 32 + lq) * KS + 16 * s + 8 * lh);
        };
        // two accumulators, where there are registers for them: a product waits for the one before the last
        v16f sacc, sodd;
#pragma unroll
        for (int r = 0; r < 16; r++) sacc[r] = sodd[r] = 0.f;
#pragma unroll
        for (uint32_t s = 0; s < NS; s += 2) {
            sacc = mma32(k_frag(s), qf[s], sacc);
            if constexpr (FOUR) sacc = mma32(k_frag(s + 1), qf[s + 1], sacc);
            else sodd = mma32(k_frag(s + 1), qf[s + 1], sodd);
        }
        if constexpr (!FOUR) {
#pragma unroll
            for (int r = 0; r < 16; r++) sacc[r] = DIRECT ? sacc[r] + sodd[r] : (sacc[r] + sodd[r]) * c2;
        }
        if (k0 + 31 > wave_min || k0 < last_lo) {
#pragma unroll
            for (int r = 0; r < 16; r++) {
                const uint32_t t = k0 + 8 * (r >> 2) + 4 * lh + (r & 3);
                sacc[r] = (t <= qpos && qpos - t < window) ? sacc[r] : -INFINITY;
            }
        }
        float m_tile = sacc[0];
#pragma unroll
        for (int r = 1; r < 16; r++) m_tile = fmaxf(m_tile, sacc[r]);
        m_tile = lane_xor_max<32>(m_tile) * later;
        const bool risen = m_tile > m_run;
        if (__builtin_amdgcn_ballot_w64(risen) != 0) {
            const float m_new = risen ? m_tile : m_run;
            const float alpha = m_run == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m_run - m_new);
            l_run *= alpha;
#pragma unroll
            for (uint32_t d = 0; d < ND; d++)
#pragma unroll
                for (int r = 0; r < 16; r++) oacc[d][r] *= alpha;
            m_run = m_new;
        }
        const float m_exp = m_run == -INFINITY ? 0.f : m_run;            // no key seen yet: every weight is 2^-inf = 0
        x8 pb[2];
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int e = 0; e < 8; e++) {
                const float p = __builtin_amdgcn_exp2f(fmaf(sacc[8 * j + e], later, -m_exp));
                l_run += p;
                pb[j][e] = (T)p;
            }
        // element e of lane half lh is key 16 j + 8 (e / 4) + 4 lh + e % 4 of the wave's half
        if constexpr (DIRECT) {
            constexpr int N = ND > 1 ? 2 : 1;
            const uint32_t base = (uint32_t)(uintptr_t)FH_LDS3(pair);
#pragma unroll
            for (uint32_t d = 0; d < ND; d += N) {
                v8bf vf[2][N];
                read_v<N, CHUNK>(vf, base + v_at + d * CHUNK, base + (v_at ^ 32) + 512 + d * CHUNK);
#pragma unroll
                for (int j = 0; j < 2; j++)
#pragma unroll
                    for (int i = 0; i < N; i++) oacc[d + i] = mma32(vf[j][i], pb[j], oacc[d + i]);
            }
        } else {
#pragma unroll
            for (int j = 0; j < 2; j++)
#pragma unroll
                for (uint32_t d = 0; d < ND; d++) {
                    const T* vr = Vt + (d * 32 + lq) * VS + kh * 32 + 16 * j + 4 * lh;
                    const x4 v0 = *reinterpret_cast<const x4*>(vr), v1 = *reinterpret_cast<const x4*>(vr + 8);
                    oacc[d] = mma32((x8){v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]}, pb[j], oacc[d]);
                }
        }
    }

    // ---- merge: the first wave of a group takes the states of the others through LDS, 32 output columns at a time
    float* mg = reinterpret_cast<float*>(ap_lds) + (qg * (KG - 1) * 64 + lane) * 18;      // wave k of the group: + (k - 1) 64 18
    float* mine = mg + (kh - 1) * (64 * 18);
    __syncthreads();
    if (kh) { mine[16] = m_run; mine[17] = l_run; }
    __syncthreads();
    float m_all = m_run;                                                   // finite for rows < M: a query sees itself
#pragma unroll
    for (int k = 0; k < KG - 1; k++) m_all = fmaxf(m_all, mg[k * (64 * 18) + 16]);
    const float m_ref = m_all == -INFINITY ? 0.f : m_all;
    const float a0 = __builtin_amdgcn_exp2f(m_run - m_ref);
    float a1[KG - 1], l_all = l_run * a0;
#pragma unroll
    for (int k = 0; k < KG - 1; k++) {
        a1[k] = __builtin_amdgcn_exp2f(mg[k * (64 * 18) + 16] - m_ref);
        l_all += mg[k * (64 * 18) + 17] * a1[k];
    }
    const float inv = 1.0f / lane_xor_add<32>(l_all);
#pragma unroll
    for (uint32_t d = 0; d < ND; d++) {
        if (kh) {
#pragma unroll
            for (int r = 0; r < 16; r++) mine[r] = oacc[d][r];
        }
        __syncthreads();
        if (!kh && qrow < M) {
#pragma unroll
            for (int g = 0; g < 4; g++) {
                const uint32_t c = 32 * d + 8 * g + 4 * lh;
                if (c >= sh.vdim) continue;
                const size_t at = (size_t)qrow * ld_out + head * sh.vdim + c;
                const x4 gt = *reinterpret_cast<const x4*>(gate + at);
                float o[4];
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    float v = oacc[d][4 * g + i] * a0;
#pragma unroll
                    for (int k = 0; k < KG - 1; k++) v = v + mg[k * (64 * 18) + 4 * g + i] * a1[k];
                    o[i] = v * inv * (float)gt[i];
                }
                store4<T>(out + at, o[0], o[1], o[2], o[3]);
            }
        }
        __syncthreads();
    }
}

namespace {

template <typename T, int DQ, int DV, int KG>
void go_keys(const PromptAttn& a, uint32_t M, uint32_t base_pos, hipStream_t s) {
    constexpr uint32_t lds = prompt_lds<T, DQ, DV, KG>(), QB = 32 * (8 / KG);
    static_assert(lds <= 160 * 1024, "LDS of a compute unit");
    static const hipError_t ok = hipFuncSetAttribute((const void*)attn_prompt_kernel<T, DQ, DV, KG>, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    (void)ok;
    fh::launch(attn_prompt_kernel<T, DQ, DV, KG>, dim3((M + QB - 1) / QB * a.heads), LP_THREADS, lds, s, a, (const T*)a.q, (const T*)a.k, (const T*)a.v,
               (const T*)a.shared, (const T*)a.gate, (T*)a.out, M, base_pos);
}

template <typename T, int DQ, int DV>
void go(const PromptAttn& a, uint32_t M, uint32_t base_pos, hipStream_t s) {
    // Bound by the chain of tile steps (about 1.1 us each), not by work, as long as the workgroups are few: four waves to a query group while the workgroups of
    // 64 queries are a few rounds of the chip, fewer under a window, which makes them all equally long, than without, where the short ones fill the gaps.  us, two / four, by workgroups
    // of 64 queries:
    //   bfloat16, up to 96 columns (two workgroups run on a compute unit)    window 135 21.8 / 15.2, 360 27.4 / 23.3, 480 23.5 / 24.0, 567 29.7 / 32.9, 640 26.2 / 29.0; none 360 40.2 / 29.1, 480
    //                         49.6 / 34.4, 608 24.3 / 23.7, 756 78.0 / 65.7, 768 30.2 / 30.6, 1280 54.0 / 63.2
    //   128 columns (tiles of 128 keys are 128 KB, one workgroup)            window 240 22.6 / 19.3, 360 30.2 / 29.6, 576 37.7 / 50.9; none 240 22.7 / 18.9, 360 29.9 / 29.7, 456 36.6 / 38.2
    //   32-bit, 64 columns (one as well)                                     window 192 31.6 / 24.1, 256 31.3 / 24.6, 320 32.3 / 45.4; none 360 57.0 / 37.3, 480 77.5 / 60.4, 608 98.7 / 102
    // Shapes whose tiles of 128 keys do not fit stay with two, and so do up to 64 keys, one tile for two waves: four would only load and merge more (2 tokens 6.1 / 6.6 us).
    constexpr uint32_t CUS = 256;
    const bool windowed = a.window && a.window < base_pos + M;
    const uint32_t at_most = prompt_four<T, DQ>() ? (windowed ? 2 * CUS : 3 * CUS - 1) : sizeof(T) == 2 ? (windowed ? CUS : CUS * 3 / 2) : (windowed ? CUS : 2 * CUS);
    if constexpr (sizeof(T) == 2 ? DQ <= 128 : prompt_lds<T, DQ, DV, 4>() <= 80 * 1024)
        if (base_pos + M > 64 && (uint64_t)((M + 63) / 64) * a.heads <= at_most) { go_keys<T, DQ, DV, 4>(a, M, base_pos, s); return; }
    go_keys<T, DQ, DV, 2>(a, M, base_pos, s);
}

template <typename T>
void by_size(const PromptAttn& a, uint32_t M, uint32_t base_pos, hipStream_t s) {
    const uint32_t dq = a.dim + a.rot, dv = a.vdim;
#define FH_AP(DQ_, DV_) if (dq <= DQ_ && dv <= DV_) { go<T, DQ_, DV_>(a, M, base_pos, s); return; }
    FH_AP(64, 32)
    FH_AP(64, 64)
    FH_AP(96, 64)
    FH_AP(128, 128)
    FH_AP(192, 128)
    FH_AP(256, 256)
#undef FH_AP
}

}  // namespace

void launch_attn_prompt(DType t, const PromptAttn& a, uint32_t M, uint32_t base_pos, hipStream_t s) {
    if (t == DType::BF16) by_size<__bf16>(a, M, base_pos, s);
    else by_size<float>(a, M, base_pos, s);
}

}  // namespace fh
