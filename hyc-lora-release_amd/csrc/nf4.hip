// NF4 (4-bit NormalFloat) block-wise weight dequantisation for gfx950, bitsandbytes 0.43 layout.
//
// The reference keeps its frozen weights as bitsandbytes NF4 with double quantisation and turns
// them into dense bf16 with BF.dequantize_nf4 on every use (models/utils/compute_utils.py:19, :29).
// Format (bitsandbytes/functional.py dequantize_4bit, csrc/kernels.cu kDequantizeBlockwise):
//   * two codes per byte, the element with the EVEN index in the high nibble;
//   * value = table[code] * absmax[element / blocksize], an fp32 product rounded to the output type;
//   * nested ("double quant") statistics: absmax[b] = code2[absmax_code[b]] * absmax2[b / blocksize2]
//     + offset, all fp32 (dequantize_blockwise followed by `absmax += offset`; offset is a device scalar).
// One lane turns 4 packed bytes into one 16-byte chunk of 8 bf16 values, kNf4Chunks of them with all loads ahead; the two
// tables sit in LDS.  HBM-bound: 0.5 + 2 bytes per element.  One chunk a lane with two 64-bit divisions by the block sizes and the
// statistics' table read from memory behind its code took 33 us for [11008, 4096] where the bytes take 19; block sizes are powers of
// two in every checkpoint there is and become shifts, others keep a division.  19 us now, 9.7 -> 8.8 for [4096, 4096].  The stores are
// ordinary ones although the weight is written once: the product that follows reads it back.  Non-temporal they take 1 us less and the
// product more: 179 against 177 us for dequantisation and product at 2048 x 4096 x 11008, 274 against 239 at 2048 x 5120 x 13824.
#include "hyc_common.hpp"

namespace hyc {

constexpr int kNf4Threads = 256;
constexpr int kNf4Chunks = 4;

struct Nf4Args {
    const uint8_t* packed; const void* absmax; const float* code2; const float* absmax2; const float* offset; const float* table;
    uint16_t* out;
    int64_t n;
    int blocksize, blocksize2, shift, shift2;      // the shifts where both are powers of two
};

template <bool NESTED, bool POW2>
__global__ __launch_bounds__(kNf4Threads) void nf4_dequant_kernel(const Nf4Args a) {
    __shared__ float tbl[16];
    __shared__ float stat[NESTED ? 256 : 1];
    const int64_t chunk0 = (int64_t)blockIdx.x * (kNf4Threads * kNf4Chunks) + threadIdx.x;
    const int64_t last = a.n / 8 - (a.n % 8 == 0 ? 1 : 0);      // last chunk, whole or not
    uint32_t w[kNf4Chunks], code[kNf4Chunks];
    float am[kNf4Chunks], am2[kNf4Chunks];
#pragma unroll
    for (int k = 0; k < kNf4Chunks; ++k) {
        const int64_t chunk = chunk0 + k * kNf4Threads < last ? chunk0 + k * kNf4Threads : last;
        // blocksize % 8 == 0: a chunk never straddles blocks
        const int64_t blk = POW2 ? (chunk * 8) >> a.shift : chunk * 8 / a.blocksize;
        if constexpr (NESTED) {
            code[k] = ((const uint8_t*)a.absmax)[blk];
            am2[k] = a.absmax2[POW2 ? blk >> a.shift2 : blk / a.blocksize2];
        } else {
            am[k] = ((const float*)a.absmax)[blk];
        }
        w[k] = chunk * 8 + 8 <= a.n ? *reinterpret_cast<const uint32_t*>(a.packed + chunk * 4) : 0u;
    }
    const float offset = NESTED && a.offset ? *a.offset : 0.0f;
    if (threadIdx.x < 16) tbl[threadIdx.x] = a.table[threadIdx.x];
    if constexpr (NESTED) stat[threadIdx.x] = a.code2[threadIdx.x];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < kNf4Chunks; ++k) {
        const int64_t e0 = (chunk0 + k * kNf4Threads) * 8;
        if constexpr (NESTED) am[k] = stat[code[k]] * am2[k] + offset;
        if (e0 + 8 <= a.n) {
            float f[8];
#pragma unroll
            for (int b = 0; b < 4; ++b) {
                const uint32_t byte = (w[k] >> (8 * b)) & 0xffu;
                f[2 * b] = tbl[byte >> 4] * am[k];
                f[2 * b + 1] = tbl[byte & 15u] * am[k];
            }
            st16(a.out + e0, pack8(f));
        } else if (e0 < a.n) {
            for (int j = 0; e0 + j < a.n; ++j) {
                const uint32_t byte = a.packed[(e0 + j) / 2];
                a.out[e0 + j] = f_to_bf(tbl[j & 1 ? byte & 15u : byte >> 4] * am[k]);
            }
        }
    }
}

}  // namespace hyc

using namespace hyc;

extern "C" int hyc_nf4_dequant(const void* packed, const void* absmax, int nested, const float* code2,
                               const float* absmax2, const float* offset, int64_t blocksize2, const float* table, void* out,
                               int64_t n, int64_t blocksize, void* stream) {
    if (n < 0 || blocksize <= 0 || blocksize % 8 != 0 || n % 2 != 0) return HYC_ERR_SHAPE;
    if (nested && blocksize2 <= 0) return HYC_ERR_SHAPE;
    if (n == 0) return HYC_OK;
    if (!packed || !absmax || !table || !out || (nested && (!code2 || !absmax2))) return HYC_ERR_NULL;
    if ((reinterpret_cast<uintptr_t>(packed) & 3u) || !aligned16(out)) return HYC_ERR_ALIGN;
    const int64_t blocks = cdiv(cdiv(n, (int64_t)8), (int64_t)kNf4Threads * kNf4Chunks);
    if (blocks > INT32_MAX || blocksize > INT32_MAX || (nested && blocksize2 > INT32_MAX)) return HYC_ERR_SHAPE;
    Nf4Args a{(const uint8_t*)packed, absmax, code2, absmax2, offset, table, (uint16_t*)out, n, (int)blocksize, nested ? (int)blocksize2 : 1, 0, 0};
    auto pow2 = [](int64_t v) { return (v & (v - 1)) == 0; };
    const bool shifts = pow2(a.blocksize) && pow2(a.blocksize2);
    a.shift = __builtin_ctz((unsigned)a.blocksize);
    a.shift2 = __builtin_ctz((unsigned)a.blocksize2);
    const dim3 grid((unsigned)blocks), block(kNf4Threads);
    hipStream_t st = (hipStream_t)stream;
    if (nested && shifts) hipLaunchKernelGGL((nf4_dequant_kernel<true, true>), grid, block, 0, st, a);
    else if (nested) hipLaunchKernelGGL((nf4_dequant_kernel<true, false>), grid, block, 0, st, a);
    else if (shifts) hipLaunchKernelGGL((nf4_dequant_kernel<false, true>), grid, block, 0, st, a);
    else hipLaunchKernelGGL((nf4_dequant_kernel<false, false>), grid, block, 0, st, a);
    return check_launch();
}
