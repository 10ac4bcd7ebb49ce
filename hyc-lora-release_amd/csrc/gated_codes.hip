// The gated product of an MLP whose layer keeps every activation as codes ('intra' layers), for gfx950:
//
//   forward   fn = bf16(silu(gate)), out = bf16(up * fn);  codes of gate, up, fn and out      (reference:
//             fused_llama_layer_intra.py:234-255: F.silu, a product and four quantisers, seven passes)
//   backward  from the codes of gate, up and fn:  grad_up = bf16(grad * fn),  grad_gate = silu_backward(gate, bf16(grad * up))
//             (:330-362: three dequantisers, two products and silu_backward, six passes)
//
// Operation by operation the values of the separate passes (silu as torch evaluates it, silu_backward of elementwise.hip, the code
// rule of quant_pack.hip).  A lane keeps one chunk of 8 columns and walks down rows, as there; the next row's operands are requested before
// the current one is worked on.  Bound by memory and, forward, as much by instructions: 4 quantisers of about 8 an element and an exponential
// and a division.  [2040, 13824] at 8 bits, us: forward 110 for the separate passes -> 60, backward 150 -> 68 (4.7 and 3.7 TB/s).
#include <type_traits>

#include "hyc_pack.hpp"

namespace hyc {

constexpr int kGcThreads = 256;
constexpr int kGcWaves = kGcThreads / kWave;

struct GatedCodesArgs {
    const uint16_t *gate, *up, *grad;
    uint16_t *out, *out2;                // forward: the product; backward: gradients of gate and up
    const uint16_t* s[4];                // steps of gate, up, fn, product
    uint8_t* q[4];
    int64_t T;
    int N, C, col_tiles, rows;               // rows a wave walks
};

// Which lane has which chunk, and its rows
struct GatedCodesPlace {
    int chunk, ld_chunk;
    bool active;
    int64_t row0, row1;
    __device__ __forceinline__ explicit GatedCodesPlace(const GatedCodesArgs& a) {
        const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
        const int64_t row_tile = blockIdx.x / a.col_tiles;
        chunk = (int)(blockIdx.x - row_tile * a.col_tiles) * kWave + lane;
        active = chunk < a.C;
        ld_chunk = active ? chunk : a.C - 1;
        row0 = (row_tile * kGcWaves + wave) * a.rows;
        row1 = row0 + a.rows < a.T ? row0 + a.rows : a.T;
    }
};

template <int QBIT>
__global__ __launch_bounds__(kGcThreads) void gated_codes_fwd_kernel(const GatedCodesArgs a) {
    const GatedCodesPlace p(a);
    if (p.row0 >= p.row1) return;
    QuantCols<QBIT> qc[4];
    bool fast = true;
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        qc[k].load(a.s[k], p.chunk * 8, p.active);
        fast = fast && qc[k].fast;
    }
    const int row_bytes = a.N / 8 * QBIT;               // (the product first would pass 2^31 at 2^28 channels)
    auto run = [&](auto fast_tag) __attribute__((always_inline)) {
        constexpr bool FAST = decltype(fast_tag)::value;
        const float zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
        u32x4 g = ld16_nt(a.gate + p.row0 * a.N + p.ld_chunk * 8), u = ld16_nt(a.up + p.row0 * a.N + p.ld_chunk * 8);
        for (int64_t t = p.row0; t < p.row1; ++t) {
            float f[4][8];
            unpack8(g, f[0]);
            unpack8(u, f[1]);
            const int64_t next = t + 1 < p.row1 ? t + 1 : t;
            g = ld16_nt(a.gate + next * a.N + p.ld_chunk * 8);
            u = ld16_nt(a.up + next * a.N + p.ld_chunk * 8);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                f[2][j] = rbf(f[0][j] / (1.0f + expf(-f[0][j])));
                f[3][j] = f[1][j] * f[2][j];
            }
            const u32x4 o = pack8(f[3]);
            unpack8(o, f[3]);
            if (p.active) st16(a.out + t * a.N + p.chunk * 8, o);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                uint32_t lo, hi;
                codes_to_words<QBIT, false, FAST>(f[k], qc[k], zero, lo, hi);
                store_packed<QBIT, false>(a.q[k] + t * row_bytes, p.chunk, p.active, lo, hi);
            }
        }
    };
    if (__ballot(!fast) == 0ull) run(std::true_type{});
    else run(std::false_type{});
}

template <int QBIT>
__global__ __launch_bounds__(kGcThreads) void gated_codes_bwd_kernel(const GatedCodesArgs a) {
    const GatedCodesPlace p(a);
    if (p.row0 >= p.row1) return;
    constexpr float kHalf = (float)(1 << (QBIT - 1));
    const PackedSlot<QBIT> slot(p.ld_chunk);
    float s[3][8];
#pragma unroll
    for (int k = 0; k < 3; ++k) unpack8(ld16(a.s[k] + p.ld_chunk * 8), s[k]);
    const int row_bytes = a.N / 8 * QBIT;
    u32x2 w[3];
    u32x4 gv;
    auto request = [&](int64_t t) __attribute__((always_inline)) {
#pragma unroll
        for (int k = 0; k < 3; ++k) w[k] = ld8(a.q[k] + t * row_bytes + slot.offset);
        gv = ld16_nt(a.grad + t * a.N + p.ld_chunk * 8);
    };
    request(p.row0);
    for (int64_t t = p.row0; t < p.row1; ++t) {
        float f[3][8], g[8], og[8], ou[8];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            slot.decode(w[k], f[k]);
#pragma unroll
            for (int j = 0; j < 8; ++j) f[k][j] = rbf((f[k][j] - kHalf) * s[k][j]);
        }
        unpack8(gv, g);
        request(t + 1 < p.row1 ? t + 1 : t);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const float sig = rbf(sigmoidf_(f[0][j]));
            const float d = rbf(sig * rbf(1.0f + rbf(f[0][j] * rbf(1.0f - sig))));
            og[j] = rbf(g[j] * f[1][j]) * d;
            ou[j] = g[j] * f[2][j];
        }
        if (p.active) {
            st16(a.out + t * a.N + p.chunk * 8, pack8(og));
            st16(a.out2 + t * a.N + p.chunk * 8, pack8(ou));
        }
    }
}

static int gated_codes_prepare(GatedCodesArgs& a, const void* const* steps, void* const* codes, int count, int64_t T, int64_t N, int q_bit,
                               dim3& grid) {
    if (q_bit != 2 && q_bit != 4 && q_bit != 8) return HYC_ERR_QBIT;
    if (T < 0 || N < 0 || N % 32 != 0 || N > (1 << 28) || T > ((int64_t)1 << 40)) return HYC_ERR_SHAPE;
    if (!steps || !codes) return HYC_ERR_NULL;
    for (int k = 0; k < count; ++k) {
        if (!steps[k] || !codes[k]) return HYC_ERR_NULL;
        if (!aligned16(steps[k]) || (reinterpret_cast<uintptr_t>(codes[k]) & 7u)) return HYC_ERR_ALIGN;
        a.s[k] = (const uint16_t*)steps[k];
        a.q[k] = (uint8_t*)codes[k];
    }
    a.T = T;
    a.N = (int)N;
    a.C = (int)(N / 8);
    a.col_tiles = (int)cdiv(a.C, kWave);
    // 8 rows a wave load the steps half as often as 4, which pays once a chip full of waves (8 a SIMD) is left: forward / backward at 4 bits,
    // us: [8192, 11008] 149 / 151 against 155 / 147, [512, 11008] 21.4 / 17.9 against 18.5 / 15.8; 2 and 16 rows are slower at both.
    a.rows = T * a.col_tiles >= (int64_t)8 * 8192 ? 8 : 4;
    const int64_t wgs = cdiv(T, (int64_t)kGcWaves * a.rows) * a.col_tiles;
    if (wgs > INT32_MAX) return HYC_ERR_SHAPE;
    grid = dim3((unsigned)wgs);
    return HYC_OK;
}

}  // namespace hyc

using namespace hyc;

extern "C" int hyc_silu_mul_codes(const void* gate, const void* up, const void* const* steps, void* const* codes, void* out, int64_t T, int64_t N,
                                  int q_bit, void* stream) {
    GatedCodesArgs a{};
    dim3 grid;
    const int rc = gated_codes_prepare(a, steps, codes, 4, T, N, q_bit, grid);
    if (rc != HYC_OK || T * N == 0) return rc;
    if (!gate || !up || !out) return HYC_ERR_NULL;
    if (!aligned16(gate) || !aligned16(up) || !aligned16(out)) return HYC_ERR_ALIGN;
    a.gate = (const uint16_t*)gate; a.up = (const uint16_t*)up; a.out = (uint16_t*)out;
    hipStream_t st = (hipStream_t)stream;
    if (q_bit == 8) hipLaunchKernelGGL(gated_codes_fwd_kernel<8>, grid, dim3(kGcThreads), 0, st, a);
    else if (q_bit == 4) hipLaunchKernelGGL(gated_codes_fwd_kernel<4>, grid, dim3(kGcThreads), 0, st, a);
    else hipLaunchKernelGGL(gated_codes_fwd_kernel<2>, grid, dim3(kGcThreads), 0, st, a);
    return check_launch();
}

extern "C" int hyc_silu_mul_bwd_codes(const void* const* codes, const void* const* steps, const void* grad, void* grad_gate, void* grad_up, int64_t T,
                                      int64_t N, int q_bit, void* stream) {
    GatedCodesArgs a{};
    dim3 grid;
    const int rc = gated_codes_prepare(a, steps, const_cast<void* const*>(codes), 3, T, N, q_bit, grid);
    if (rc != HYC_OK || T * N == 0) return rc;
    if (!grad || !grad_gate || !grad_up) return HYC_ERR_NULL;
    if (!aligned16(grad) || !aligned16(grad_gate) || !aligned16(grad_up)) return HYC_ERR_ALIGN;
    a.grad = (const uint16_t*)grad; a.out = (uint16_t*)grad_gate; a.out2 = (uint16_t*)grad_up;
    hipStream_t st = (hipStream_t)stream;
    if (q_bit == 8) hipLaunchKernelGGL(gated_codes_bwd_kernel<8>, grid, dim3(kGcThreads), 0, st, a);
    else if (q_bit == 4) hipLaunchKernelGGL(gated_codes_bwd_kernel<4>, grid, dim3(kGcThreads), 0, st, a);
    else hipLaunchKernelGGL(gated_codes_bwd_kernel<2>, grid, dim3(kGcThreads), 0, st, a);
    return check_launch();
}
