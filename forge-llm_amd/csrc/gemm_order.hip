// Quantised matmul for a few rows of activations in the order-faithful mode (matmul_mat_q8_0_KxN / matmul_mat_q4_0_KxN, emit.rs:2108-2302,
// 3667-3817): r += (a_scale * w_scale) * f32(isum), block by block, nothing fused, for every result on its own.
//
// What bounds it: the chain along K.  A result's blocks cannot be shared out, so what is left is to make a block's step short and to spread
// the results: a wave works 16 x 16 of them, one v_mfma_i32_16x16x32_i8 (K = 32 is one quant block) and sixteen VALU instructions per block
// (convert, scale, multiply, add for the four sums of a lane), with the steps of four blocks that follow already on their way.
// The tile kernel (gemm.hip) walks K in stages of 1.25 to 2.2 us for 128 columns at a time, which leaves most of the chip idle for a narrow
// matrix.  33 rows with the quantiser, us: 576 -> 576 16.7 -> 7.6, 2048 -> 2048 35.7 -> 11.4, 8192 -> 2048 126 -> 28, Q4_0 3072 -> 1024 54.4 -> 15.5.
// (The scale products a_s * w_s are exact in f32, 11-bit by 11-bit significands, so it does not matter how they are made.)
#include <algorithm>

#include "common.h"
#include "device_utils.h"

namespace fh {

namespace {

typedef int v4i __attribute__((ext_vector_type(4)));

constexpr int GO_U = 4;                      // blocks of a step: 128 bytes of a Q8_0 or activation row, 64 of a Q4_0 row
constexpr int GO_AHEAD = 4;                  // steps in flight
constexpr uint32_t GO_RSRC = 0x00020000;     // raw buffer, 32-bit data format

struct OrderArgs {
    const uint8_t* wq;
    const uint16_t* wsc;
    const int8_t* aq;
    const uint16_t* asc;
    float* y;
    uint32_t M, N, K, ldy, accumulate;
};

template <bool Q4>
__global__ __launch_bounds__(256) void gemm_order_kernel(OrderArgs a) {
    constexpr uint32_t WB = Q4 ? 64 : 128;                     // bytes of a weight row in a step
    constexpr uint32_t LA = 16 * 128, LB = 16 * WB, STRIP = LA + LB + 512;
    __shared__ __attribute__((aligned(16))) uint8_t lds[4 * 2 * STRIP];
    const uint32_t lane = threadIdx.x & 63, wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const uint32_t c = lane & 15, g = lane >> 4;               // row (of A) / column (of B) of the operands; which 8 of a block's 32 elements
    const uint32_t nblk = a.K / 32, m0 = blockIdx.y * 16, n0 = (blockIdx.x * 4 + wave) * 16;
    if (n0 >= a.N) return;                                     // (no barrier: a wave's strip is its own)
    uint8_t* strips = lds + wave * 2 * STRIP;
    // rows past the end read as zero
    const __amdgpu_buffer_rsrc_t rw = __builtin_amdgcn_make_buffer_rsrc((void*)a.wq, 0, a.N * nblk * (Q4 ? 16 : 32), GO_RSRC);
    const __amdgpu_buffer_rsrc_t rws = __builtin_amdgcn_make_buffer_rsrc((void*)a.wsc, 0, a.N * nblk * 2, GO_RSRC);
    const __amdgpu_buffer_rsrc_t ra = __builtin_amdgcn_make_buffer_rsrc((void*)a.aq, 0, a.M * a.K, GO_RSRC);
    const __amdgpu_buffer_rsrc_t ras = __builtin_amdgcn_make_buffer_rsrc((void*)a.asc, 0, a.M * nblk * 2, GO_RSRC);
    // A step's codes go through LDS: fetched as whole 128-byte (Q4_0: 64-byte) pieces of rows and laid down in 16-byte pieces XOR-swizzled by the
    // row; fetched as operands, eight bytes of sixteen rows at a time, the memory pipe took 300 ns a block.  The scales go the same way, as floats.
    constexpr int NB = Q4 ? 1 : 2;
    const uint32_t ar = lane >> 3, ap = lane & 7, br = Q4 ? lane >> 2 : ar, bp = Q4 ? lane & 3 : ap;
    const uint32_t a_off = (m0 + ar) * a.K + ap * 16, w_off = (n0 + br) * nblk * (Q4 ? 16 : 32) + bp * 16;
    const uint32_t as_off = ((m0 + c) * nblk + g) * 2, ws_off = ((n0 + c) * nblk + g) * 2;
    struct Fetched { v4i A[2], B[NB]; uint32_t sa, sb; };
    // (what a step fetches past the end of K belongs to the next row, or reads as zero, and is not looked at)
    auto fetch = [&](Fetched& f, uint32_t st) {
#pragma unroll
        for (int i = 0; i < NB; i++) f.B[i] = __builtin_amdgcn_raw_buffer_load_b128(rw, w_off + i * 8 * nblk * 32 + st * WB, 0, 0);
#pragma unroll
        for (int i = 0; i < 2; i++) f.A[i] = __builtin_amdgcn_raw_buffer_load_b128(ra, a_off + i * 8 * a.K + st * 128, 0, 0);
        f.sa = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(ras, as_off + st * GO_U * 2, 0, 0);
        f.sb = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rws, ws_off + st * GO_U * 2, 0, 0);
    };
    auto as_float = [](uint32_t bits) { return (float)__builtin_bit_cast(_Float16, (uint16_t)bits); };
    auto lay_down = [&](const Fetched& f, uint32_t buf) {
        uint8_t* s = strips + buf * STRIP;
#pragma unroll
        for (int i = 0; i < 2; i++) *reinterpret_cast<v4i*>(s + (ar + 8 * i) * 128 + ((ap ^ ar) * 16)) = f.A[i];
#pragma unroll
        for (int i = 0; i < NB; i++) *reinterpret_cast<v4i*>(s + LA + (br + 8 * i) * WB + ((bp ^ (Q4 ? (br >> 1) & 3 : br)) * 16)) = f.B[i];
        float* sc = reinterpret_cast<float*>(s + LA + LB);
        sc[lane] = as_float(f.sa);                             // [block][row]
        sc[64 + lane] = Q4 ? as_float(f.sb) * 0.0625f : as_float(f.sb);
    };
    struct Operands { uint2 A[GO_U], B[GO_U]; float4 sa[GO_U]; float sb[GO_U]; };
    auto pick_up = [&](Operands& o, uint32_t buf) {
        const uint8_t* s = strips + buf * STRIP;
        const float* sc = reinterpret_cast<const float*>(s + LA + LB);
#pragma unroll
        for (int u = 0; u < GO_U; u++) {
            o.A[u] = *reinterpret_cast<const uint2*>(s + c * 128 + (((2 * u + (g >> 1)) ^ (c & 7)) * 16) + (g & 1) * 8);
            // Q4_0: elements 0..15 in the low nibbles of a block's 16 bytes, 16..31 in the high ones
            if (Q4) o.B[u] = *reinterpret_cast<const uint2*>(s + LA + c * 64 + ((u ^ ((c >> 1) & 3)) * 16) + (g & 1) * 8);
            else o.B[u] = *reinterpret_cast<const uint2*>(s + LA + c * 128 + (((2 * u + (g >> 1)) ^ (c & 7)) * 16) + (g & 1) * 8);
            o.sa[u] = *reinterpret_cast<const float4*>(sc + u * 16 + 4 * g);
            o.sb[u] = sc[64 + u * 16 + c];
        }
    };
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    const uint32_t sh = g < 2 ? 4u : 0u;
    auto block = [&](const Operands& o, int u) {
        uint2 b = o.B[u];
        // 16 (code - 8) of each nibble; the weight's scale is a sixteenth
        if (Q4) b = make_uint2(((b.x << sh) & 0xF0F0F0F0u) ^ 0x80808080u, ((b.y << sh) & 0xF0F0F0F0u) ^ 0x80808080u);
        const v4i isum = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, o.A[u]), __builtin_bit_cast(long, b), (v4i){0, 0, 0, 0}, 0, 0, 0);
        acc[0] = acc[0] + (o.sa[u].x * o.sb[u]) * (float)isum[0];
        acc[1] = acc[1] + (o.sa[u].y * o.sb[u]) * (float)isum[1];
        acc[2] = acc[2] + (o.sa[u].z * o.sb[u]) * (float)isum[2];
        acc[3] = acc[3] + (o.sa[u].w * o.sb[u]) * (float)isum[3];
    };
    const uint32_t full = nblk / GO_U, steps = (nblk + GO_U - 1) / GO_U;
    Fetched f[GO_AHEAD];
    Operands o[2];
#pragma unroll
    for (int i = 0; i < GO_AHEAD; i++) fetch(f[i], i);
    lay_down(f[0], 0);
    fetch(f[0], GO_AHEAD);
    pick_up(o[0], 0);
    for (uint32_t st = 0; st < steps; st += GO_AHEAD) {
#pragma unroll
        for (int i = 0; i < GO_AHEAD; i++) {
            // step st + i: the operands of the next one are picked up ahead of its products
            Fetched& next = f[(i + 1) % GO_AHEAD];
            lay_down(next, (i + 1) & 1);
            fetch(next, st + i + 1 + GO_AHEAD);
            pick_up(o[(i + 1) & 1], (i + 1) & 1);
            const Operands& now = o[i & 1];
            if (st + i < full) {
#pragma unroll
                for (int u = 0; u < GO_U; u++) block(now, u);
            } else {
#pragma unroll
                for (int u = 0; u < GO_U; u++)
                    if ((st + i) * GO_U + u < nblk) block(now, u);
            }
        }
    }
    // lane: column c, rows 4 g + r
    if (n0 + c < a.N) {
        float* y = a.y + (size_t)(m0 + 4 * g) * a.ldy + n0 + c;
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (m0 + 4 * g + r < a.M) y[(size_t)r * a.ldy] = a.accumulate ? y[(size_t)r * a.ldy] + acc[r] : acc[r];
    }
}

}  // namespace

// 32-bit byte offsets, a grid of two dimensions, and an estimate of both kernels in microseconds.  Here: rounds of 256 workgroups of 16 rows by 64
// columns, each 1.5 + 2.95 per 1024 of depth.  The tile kernel: stages of 128 of depth at 1.25 for 64-row tiles (more than 64 rows, no more of
// those tiles than CUs), 2.2 for each round of 128-row tiles.  Measured with the quantiser, tiles / this, Q8_0: 2048 -> 8192 by 2 rows 36.1 / 11.0, 64
// 36.3 / 19.9, 65 24.8 / 26.8 (stays on the tiles); 8192 -> 2048 by 33 126 / 28, 256 85.5 / 57.4, 352 87.5 / 79.1, 450 89.4 / 101; 576 -> 576 by 300 12.2 / 8.1,
// 576 -> 1536 by 300 12.7 / 11.1, 352 12.5 / 14.1; 2048 -> 512 by 902 27.3 / 21.6.
bool gemm_order_pays(const QWeight& w, uint32_t M) {
    const uint64_t limit = 0x7FFFFFFFull - 65536;
    if (M > 65535u * 16u || (uint64_t)M * w.K > limit || (uint64_t)w.N * std::max<uint64_t>(w.qs_row_bytes(), w.K / 16) > limit) return false;
    auto up = [](uint64_t n, uint64_t by) { return (n + by - 1) / by; };
    const double order = 2.0 + up(up(w.N, 64) * up(M, 16), 256) * (1.5 + 2.95 * w.K / 1024.0);
    const bool low = M > 64 && up(w.N, 128) * up(M, 64) <= 256;
    const double tiles = 3.0 + up(w.K, 128) * (low ? 1.25 : 2.2 * up(up(w.N, 128) * up(M, 128), 256));
    return order < tiles;
}

void launch_gemm_order(const QWeight& w, const int8_t* aq, const uint16_t* as, uint32_t M, float* y, uint32_t ldy, bool accumulate, hipStream_t s) {
    const OrderArgs a{w.qs, w.scales, aq, as, y, M, w.N, w.K, ldy, accumulate ? 1u : 0u};
    const dim3 grid((w.N + 63) / 64, (M + 15) / 16);
    if (w.wdtype == FORGE_HIP_Q4_0) fh::launch(gemm_order_kernel<true>, grid, 256, 0, s, a);
    else fh::launch(gemm_order_kernel<false>, grid, 256, 0, s, a);
}

}  // namespace fh
