// Projections with a frozen weight and a LoRA adapter in one pass, for gfx950, at the sizes where a library product and the
// passes around it are bound by launches and by reading the product again:
//
//   main = bf16( x W^T [+ bias] ) or bf16( x W )         (W [N, K] as nn.Linear keeps it; input gradients take it as [K, N])
//   plain    :  y = bf16(main + bf16(xa . b))  [ gelu ]  [ then y = bf16(residual + y) ]
//   quantise :  q = pack(code(main; s)),  y as above
//   sum      :  y = t_0 (+) t_1 (+) t_2 [(+) residual],  t_i = the plain form of projection i, every (+) a bf16 addition in that order
//
// which is lora_forward / lora_backward of the reference (models/utils/compute_utils.py:18-36) with what follows them in the
// layers (models/roberta/fused_roberta_layer_intra_inter.py:90-121, :355-420): bias, codes of the frozen part, the
// LoRA add, the activation, the residual, the sum of the input gradients of projections that share their input.  The arithmetic
// after the product is that of lora_add.hip.
//
// A workgroup of 4 waves forms 128 x 128 results, 64 x 64 a wave, as products of 16x16x32 along the contraction from its start to its
// end, which is also the order of the library's kernels for these sizes: same bits in every case compared, but for 3 of 10000 results
// with few tiles and a long contraction, which the library splits.  The operands come through
// LDS in tiles of 64 along the contraction (hyc_attn_tile.hpp), the copies of the next one under way; a turn takes 0.65 us, which is its
// LDS reads (96 KB a workgroup) where two workgroups share a unit and cover each other's waits (from 257 tiles on), and its waits where a
// unit has one.  (Four stages with three tiles on the
// way and one workgroup a unit: 18 against 16 us at 4096 x 768 x 768, 50 against 36 for three members.)  The product is formed transposed, so
// that a lane holds four neighbouring columns of a row, and goes through LDS once more, rounded, into the ownership of the packed
// codes: a lane has 8 consecutive columns of four rows.  Several projections of one x go into one launch.
// us, against the library's product with bias add and LoRA add with codes (x A apart): [4096, 768] x 768 16 / 27, three members 36 / 82;
// x 3072 36 / 52; [4096, 3072] x 768 41 / 40; input gradients: 768 x 768 12.5 / 20, three members 30 / 51; 3072 x 768 35 / 42, 768 x
// 3072 30 / 34.
#include <type_traits>

#include "hyc_attn_tile.hpp"
#include "hyc_lora_tile.hpp"

namespace hyc {

constexpr int kGemmThreads = 256;
constexpr int kGemmTile = 128;                     // rows and columns of a workgroup
constexpr int kGemmK = 64;                         // of the contraction at a time
constexpr int kGemmPitch = kGemmTile + 8;          // LDS row pitch of the rounded product
constexpr int kGemmMembers = 3;

struct GemmMember {
    const uint16_t *x, *w, *xa, *b, *bias, *res, *s;
    uint8_t* q;
    uint16_t* y;
    int N, K, b_transposed, cols, first_wg;        // cols: column tiles
};
struct GemmArgs {
    GemmMember m[kGemmMembers];
    int members, wgs, T, R, gelu;
};

// lane's address parts in tiles of the two forms: rows of the contraction together (x, W [N, K]) or its columns (W [K, N])
struct GemmLane {
    uint32_t row, col[2][2];
    __device__ __forceinline__ explicit GemmLane(int lane) {
        typedef AttnTile<kGemmK, kGemmTile> X;
        const int i = lane & 15, g = lane >> 4;
        row = (uint32_t)X::in_block(i, g);
#pragma unroll
        for (int odd = 0; odd < 2; ++odd)
#pragma unroll
            for (int half = 0; half < 2; ++half) {
                const int r = 8 * (g & 1) + 4 * half + (i >> 2), c = 2 * odd + ((i & 3) >> 1);
                // k rows 32 and more apart are whole blocks; of a step's 32 rows, g / 2 is the block
                col[odd][half] = (uint32_t)((g >> 1) * (kGemmTile / 32) * 1024 + X::in_block(r, c) + (i & 1) * 8);
            }
    }
};

__device__ __forceinline__ float gelu_erf(float x) { return x * 0.5f * (1.0f + erff(x * 0.70710678118654752440f)); }

// main tile of one projection: rows row0 .. +127, columns col0 .. +127, rounded into LDS
template <bool KN, bool BIAS>
__device__ __forceinline__ void gemm_tile(const GemmMember& m, int T, int row0, int col0, char* lds, uint32_t lds0, const GemmLane& at, int wave, int lane) {
    using X = AttnTile<kGemmK, kGemmTile>;
    using W = std::conditional_t<KN, AttnTile<kGemmTile, kGemmK>, AttnTile<kGemmK, kGemmTile>>;
    constexpr int kStage = X::kBytes + W::kBytes;
    const int wr = wave >> 1, wc = wave & 1;
    uint32_t off_x[X::kCopies], off_w[W::kCopies];
#pragma unroll
    for (int i = 0; i < X::kCopies; ++i) off_x[i] = X::source(i * 4 + wave, row0, T - 1, m.K, lane);
#pragma unroll
    for (int i = 0; i < W::kCopies; ++i) off_w[i] = KN ? W::source(i * 4 + wave, 0, 0x7fffffff, m.N, lane) : W::source(i * 4 + wave, col0, 0x7fffffff, m.K, lane);
    const uint16_t* x = m.x;
    const uint16_t* w = KN ? m.w + col0 : m.w;
    const int64_t w_step = KN ? (int64_t)kGemmK * m.N : kGemmK;
    const int turns = m.K / kGemmK;
    auto request = [&](int stage) {
        const uint32_t to = lds0 + (uint32_t)(stage * kStage + wave * 1024);
#pragma unroll
        for (int i = 0; i < X::kCopies; ++i) copy_to_lds16(x, off_x[i], to + (uint32_t)(i * 4096));
#pragma unroll
        for (int i = 0; i < W::kCopies; ++i) copy_to_lds16(w, off_w[i], to + (uint32_t)(X::kBytes + i * 4096));
        x += kGemmK;
        w += w_step;
    };
    f32x4 acc[4][4];                                // [16 columns][16 rows]: lane (i, g) has row i, columns 4g .. +3
#pragma unroll
    for (int a = 0; a < 4; ++a)
#pragma unroll
        for (int b = 0; b < 4; ++b) acc[a][b] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    typedef const __attribute__((address_space(3))) u32x4 lds_u32x4;
    typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
    request(0);
    for (int turn = 0; turn < turns; ++turn) {
        wait_copies_and_barrier();
        if (turn + 1 < turns) request((turn + 1) & 1);
        const uint32_t tile = lds0 + (uint32_t)((turn & 1) * kStage);
        const uint32_t in_x = tile + at.row + (uint32_t)(wr * 4 * X::kBlocksAcross * 1024);
        const uint32_t in_w = tile + X::kBytes;
#pragma unroll
        for (int ks = 0; ks < 2; ++ks) {
            bf16x8 xo[4], wo[4];
#pragma unroll
            for (int b = 0; b < 4; ++b) xo[b] = as_bf16x8(*(lds_u32x4*)(in_x + (uint32_t)((b * X::kBlocksAcross + ks) * 1024)));
#pragma unroll
            for (int a = 0; a < 4; ++a) {
                if constexpr (KN) {
                    const uint32_t blk = in_w + (uint32_t)((2 * ks * W::kBlocksAcross + wc * 2 + a / 2) * 1024);
                    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(blk + at.col[a & 1][0]));
                    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(blk + at.col[a & 1][1]));
                    const u32x2 l = __builtin_bit_cast(u32x2, lo), h = __builtin_bit_cast(u32x2, hi);
                    wo[a] = as_bf16x8(u32x4{l.x, l.y, h.x, h.y});
                } else {
                    wo[a] = as_bf16x8(*(lds_u32x4*)(in_w + at.row + (uint32_t)(((wc * 4 + a) * W::kBlocksAcross + ks) * 1024)));
                }
            }
#pragma unroll
            for (int a = 0; a < 4; ++a)
#pragma unroll
                for (int b = 0; b < 4; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wo[a], xo[b], acc[a][b], 0, 0, 0);
        }
    }
    __syncthreads();                                // the last tile has been read; no copy is under way
    const int i = lane & 15, g = lane >> 4;
#pragma unroll
    for (int a = 0; a < 4; ++a) {
        const int c = wc * 64 + 16 * a + 4 * g;
        float add[4] = {0.0f, 0.0f, 0.0f, 0.0f};
        if constexpr (BIAS) {
            if (m.bias) {                           // uniform
                const u32x2 bv = ld8(m.bias + col0 + c);
                add[0] = bf_lo(bv.x); add[1] = bf_hi(bv.x); add[2] = bf_lo(bv.y); add[3] = bf_hi(bv.y);
            }
        }
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            float f[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) f[e] = BIAS ? rbf(acc[a][b][e]) + add[e] : acc[a][b][e];
            *reinterpret_cast<u32x2*>(lds + ((wr * 64 + 16 * b + i) * kGemmPitch + c) * 2) = u32x2{pk_bf16(f[0], f[1]), pk_bf16(f[2], f[3])};
        }
    }
    __syncthreads();
}

// QBIT 0: no codes
template <int QBIT, bool KN, bool SUM>
__global__ __launch_bounds__(kGemmThreads, 2) void lora_gemm_kernel(const GemmArgs A) {
    constexpr int kLds = 2 * (AttnTile<kGemmK, kGemmTile>::kBytes + AttnTile<kGemmTile, kGemmK>::kBytes);
    static_assert(kGemmTile * kGemmPitch * 2 <= kLds, "the rounded product reuses the tiles");
    __shared__ __attribute__((aligned(1024))) char lds[kLds];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, g = lane >> 4;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    const GemmLane at(lane);
    // neighbouring workgroups on one XCD: they read the same x or the same W
    const int per = A.wgs / 8, rest = A.wgs % 8, xcd = blockIdx.x % 8;
    const int wg = xcd * per + min(xcd, rest) + (int)(blockIdx.x / 8);
    int mi = 0;
    if constexpr (!SUM) mi = (A.members > 1 && wg >= A.m[1].first_wg ? 1 : 0) + (A.members > 2 && wg >= A.m[2].first_wg ? 1 : 0);
    const GemmMember& m0 = A.m[mi];
    const int local = wg - m0.first_wg;
    const int row_tile = local / m0.cols, row0 = row_tile * kGemmTile, col0 = (local - row_tile * m0.cols) * kGemmTile;
    const int mine0 = row0 + wave * 32;             // the wave's rows after the product
    const int col = col0 + 8 * j, chunk = col / 8;
    constexpr int QB = QBIT ? QBIT : 8;
    u32x4 total[SUM ? 2 : 1][4];
#pragma unroll 1
    for (int k = 0; k < (SUM ? A.members : 1); ++k) {
        const GemmMember& m = A.m[SUM ? k : mi];
        // what the passes after the product need, on its way during the product
        u32x2 xa[2][1];
#pragma unroll
        for (int h = 0; h < 2; ++h) xa[h][0] = u32x2{0, 0};
        BOperand<1> B;
        if (SUM || m.xa) {                          // without an adapter: the frozen part alone
#pragma unroll
            for (int h = 0; h < 2; ++h) request_lora_a<1>(m.xa, A.R, min(mine0 + 16 * h + j, A.T - 1), g, xa[h]);
            B.load(m.b, m.N, A.R, col, true, g, m.b_transposed != 0);
        }
        QuantCols<QB> qc;
        bool fast = false;
        if constexpr (QBIT != 0) {
            qc.load(m.s, col, true);
            fast = __ballot(!qc.fast) == 0ull;
        }
        gemm_tile<KN, !SUM>(m, A.T, row0, col0, lds, lds0, at, wave, lane);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int r0 = mine0 + 16 * h;
            if (r0 >= A.T) break;                   // uniform
            uint32_t L[4][4];
            if (SUM || m.xa) {
                u32x2 xm[1];
                mask_lora_a<1>(A.R, g, xa[h], xm);
                lora_tile_bf16_regs<1>(xm, B, L);
            }
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int t = r0 + 4 * g + v;
                const bool live = t < A.T;
                float f[8], y[8];
                unpack8(*reinterpret_cast<const u32x4*>(lds + ((wave * 32 + 16 * h + 4 * g + v) * kGemmPitch + 8 * j) * 2), f);
                if constexpr (QBIT != 0) {
                    const float zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
                    uint32_t lo, hi;
                    if (fast) codes_to_words<QB, false, true>(f, qc, zero, lo, hi);
                    else codes_to_words<QB, false, false>(f, qc, zero, lo, hi);
                    store_packed<QB, false>(m.q + (int64_t)(live ? t : A.T - 1) * (m.N * QB / 8), chunk, live, lo, hi);
                }
#pragma unroll
                for (int e = 0; e < 8; ++e) y[e] = SUM || m.xa ? f[e] + lora_elem(L[v], e) : f[e];
                if constexpr (SUM) {
                    if (k) {
                        float s[8];
                        unpack8(total[h][v], s);
#pragma unroll
                        for (int e = 0; e < 8; ++e) y[e] = s[e] + rbf(y[e]);
                    }
                    total[h][v] = pack8(y);
                    if (k + 1 == A.members && live) {
                        if (m0.res) {
                            float s[8], r[8];
                            unpack8(total[h][v], s);
                            unpack8(ld16(m0.res + (int64_t)t * m.N + col), r);
#pragma unroll
                            for (int e = 0; e < 8; ++e) y[e] = s[e] + r[e];
                            total[h][v] = pack8(y);
                        }
                        st16(m0.y + (int64_t)t * m.N + col, total[h][v]);
                    }
                } else if (live) {
                    if (A.gelu) {
#pragma unroll
                        for (int e = 0; e < 8; ++e) y[e] = gelu_erf(rbf(y[e]));
                    }
                    if (m.res) {
                        float r[8];
                        unpack8(ld16(m.res + (int64_t)t * m.N + col), r);
#pragma unroll
                        for (int e = 0; e < 8; ++e) y[e] = r[e] + rbf(y[e]);
                    }
                    st16(m.y + (int64_t)t * m.N + col, pack8(y));
                }
            }
        }
        if constexpr (SUM) __syncthreads();         // the tile is read; the next projection's copies overwrite it
    }
}

template <int QBIT>
static void gemm_launch(const GemmArgs& a, bool kn, bool sum, hipStream_t st) {
    const dim3 grid((unsigned)a.wgs), block(kGemmThreads);
    if constexpr (QBIT == 0) {
        if (kn && sum) hipLaunchKernelGGL((lora_gemm_kernel<0, true, true>), grid, block, 0, st, a);
        else if (kn) hipLaunchKernelGGL((lora_gemm_kernel<0, true, false>), grid, block, 0, st, a);
        else hipLaunchKernelGGL((lora_gemm_kernel<0, false, false>), grid, block, 0, st, a);
    } else {
        hipLaunchKernelGGL((lora_gemm_kernel<QBIT, false, false>), grid, block, 0, st, a);
    }
}

}  // namespace hyc

using namespace hyc;

extern "C" int hyc_lora_gemm(const hyc_gemm_member* members, int count, int w_is_kn, int sum, int q_bit, int gelu, int64_t T, int64_t R,
                             void* stream) {
    if (!members) return HYC_ERR_NULL;
    if (count < 1 || count > kGemmMembers || (sum && !w_is_kn) || (q_bit && (w_is_kn || sum)) || (sum && gelu)) return HYC_ERR_ARG;
    if (q_bit != 0 && q_bit != 2 && q_bit != 4 && q_bit != 8) return HYC_ERR_QBIT;
    if (R < 4 || R > 16 || R % 4 != 0) return HYC_ERR_RANK;
    if (T < 1 || T > INT32_MAX - kGemmTile) return HYC_ERR_SHAPE;
    GemmArgs a{};
    a.members = count; a.T = (int)T; a.R = (int)R; a.gelu = gelu != 0;
    int64_t wgs = 0;
    for (int i = 0; i < count; ++i) {
        const hyc_gemm_member& h = members[i];
        if (h.N < kGemmTile || h.K < kGemmK || h.N % kGemmTile != 0 || h.K % kGemmK != 0) return HYC_ERR_SHAPE;
        // offsets inside an operand are 32-bit
        if (T * h.K >= (int64_t)1 << 31 || h.N * h.K >= (int64_t)1 << 31) return HYC_ERR_SHAPE;
        if (sum && h.N != members[0].N) return HYC_ERR_SHAPE;
        if (!h.x || !h.w || (sum || q_bit || gelu ? !h.xa : false) || (h.xa && !h.b) || !(sum && i ? members[0].y : h.y) || (q_bit && (!h.q || !h.scale))) return HYC_ERR_NULL;
        for (const void* p : {h.x, h.w, h.bias, h.residual, h.scale, (const void*)h.y})
            if (p && !aligned16(p)) return HYC_ERR_ALIGN;
        if ((h.xa && !(h.b_transposed ? (reinterpret_cast<uintptr_t>(h.b) & 7u) == 0 : aligned16(h.b))) || (reinterpret_cast<uintptr_t>(h.xa) & 7u) ||
            (reinterpret_cast<uintptr_t>(h.q) & 7u))
            return HYC_ERR_ALIGN;
        GemmMember& m = a.m[i];
        m.x = (const uint16_t*)h.x; m.w = (const uint16_t*)h.w; m.xa = (const uint16_t*)h.xa; m.b = (const uint16_t*)h.b;
        m.bias = (const uint16_t*)h.bias; m.res = (const uint16_t*)h.residual; m.s = (const uint16_t*)h.scale;
        m.q = (uint8_t*)h.q; m.y = (uint16_t*)h.y;
        m.N = (int)h.N; m.K = (int)h.K; m.b_transposed = h.b_transposed; m.cols = (int)(h.N / kGemmTile);
        m.first_wg = sum ? 0 : (int)wgs;
        if (!sum || i == 0) wgs += cdiv(T, kGemmTile) * m.cols;
        if (wgs > INT32_MAX) return HYC_ERR_SHAPE;
    }
    a.wgs = (int)wgs;
    hipStream_t st = (hipStream_t)stream;
    if (q_bit == 8) gemm_launch<8>(a, false, false, st);
    else if (q_bit == 4) gemm_launch<4>(a, false, false, st);
    else if (q_bit == 2) gemm_launch<2>(a, false, false, st);
    else gemm_launch<0>(a, w_is_kn != 0, sum != 0, st);
    return check_launch();
}
