// Products of a few rows with a frozen weight, on the gfx950 matrix cores:
//
//   out[t, n] = sum_k x[t, k] w[k, n]      (w [K, N]: input gradients; what the layers use, see few_rows in host/native.cpp)
//   out[t, n] = sum_k x[t, k] w[n, k]      (w [N, K]: for callers of the C entry; the layers leave x W^T to the library)
//
// Bound by the one read of w: a short batch multiplies every weight once, 2 T flops a byte.  A library product of such a
// shape gives its 256 x 256 tiles to a part of the chip.  Here the weight is cut into steps of 128 outputs x 64 of the
// contraction (16 KB), and every workgroup takes the same number of consecutive steps, whatever the shape; a workgroup's
// steps lie in at most two blocks of outputs, each of which leaves one fp32 partial sum, added up in order by a second
// kernel.  One workgroup a compute unit with the copies of the next steps (48 to 80 KB of weight) always in flight; eight waves,
// because a step is a chain of waits and addresses that four leave uncovered (39 us against 45 at 128 x 4096 x 11008).
// Steps of 64 outputs x 128 halve the partial sums and double the reads of x: 15 against 18 us at 96 x 4096 x 4096, 38
// against 31 us at 128 x 11008 x 4096.  96 rows, contraction x outputs, against the library, us: 4096 x 4096 18 / 22 forward
// and 19 / 35 backward, 11008 x 4096 30 / 50 and 29 / 85, 4096 x 11008 32 / 30 and 32 / 35; the weights take 6 and 16 us
// at the rate of a copy.  The rest are two launches, 4 us of sums, and the partial sums, which cross the fabric twice.
#include <type_traits>

#include "hyc_attn_tile.hpp"

namespace hyc {

constexpr int kFewCols = 128;          // outputs of a step: 32 per wave
constexpr int kFewK = 64;              // contraction of a step
constexpr int kFewMaxRows = 128;
constexpr int kFewUnits = 256;

struct FewArgs {
    const uint16_t *x, *w;
    float* part;                       // [workgroup][2][32 * TB][kFewCols]
    uint16_t* out;
    int T, N, K;
    int steps_k, total, groups;        // steps of a block of outputs, of all, workgroups
};

// first step of a workgroup, and the workgroup that has a step
__device__ __forceinline__ int few_first(const FewArgs& A, int group) { return (int)((int64_t)group * A.total / A.groups); }
__device__ __forceinline__ int few_group(const FewArgs& A, int step) { return (int)(((int64_t)(step + 1) * A.groups + A.total - 1) / A.total) - 1; }

// neighbouring workgroups on one XCD: they read the same x
__device__ __forceinline__ int few_logical(const FewArgs& A) {
    const int n = A.groups / 8, rest = A.groups % 8, xcd = blockIdx.x % 8, i = blockIdx.x / 8;
    return xcd * n + min(xcd, rest) + i;
}

// Stages of the copies: as many as fit beside the 16 KB of the reduction; all but one of them are in flight.
template <int TB> constexpr int kFewStages = TB <= 2 ? 6 : TB == 3 ? 5 : 4;

template <int TB, bool NK>
__global__ __launch_bounds__(512, 2) void few_rows_kernel(const FewArgs A) {
    using X = AttnTile<kFewK, 32 * TB>;
    using W = std::conditional_t<NK, AttnTile<kFewK, kFewCols>, AttnTile<kFewCols, kFewK>>;
    constexpr int kStage = X::kBytes + W::kBytes, kStages = kFewStages<TB>;
    constexpr int kXBlocks = X::kBytes / 1024, kXCopies = (kXBlocks + 7) / 8, kWCopies = 2;      // of a wave and stage
    __shared__ __attribute__((aligned(1024))) char lds[kStages * kStage + kFewCols * 32 * 4];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int wn = wave & 3, wk = wave >> 2;                                // the wave's 32 outputs and its half of a step's contraction
    const int group = few_logical(A);
    const int beg = few_first(A, group), end = few_first(A, group + 1);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    const typename X::Lane at_x(lane);
    const typename W::Lane at_w(lane);
    // what a lane copies lies at the same place of every step: offsets once, the step in the scalar base
    uint32_t off_x[kXCopies], off_w[kWCopies], to_x[kXCopies];
#pragma unroll
    for (int i = 0; i < kXCopies; ++i) {                                    // waves left over copy the last block again
        const int blk = min(i * 8 + wave, kXBlocks - 1);
        to_x[i] = (uint32_t)(blk * 1024);
        off_x[i] = X::source(blk, 0, A.T - 1, A.K, lane);
    }
#pragma unroll
    for (int i = 0; i < kWCopies; ++i) off_w[i] = W::source(i * 8 + wave, 0, 0x7fffffff, NK ? A.K : A.N, lane);
    int ks = beg % A.steps_k;                                               // of the step worked on
    int r_ks = ks, r_left = end - beg;                                      // of the next step to request
    const int64_t step = NK ? kFewK : (int64_t)kFewK * A.N;                 // a step further down the contraction
    const int64_t wrap = (NK ? (int64_t)kFewCols * A.K : kFewCols) - step * A.steps_k;          // ... and on to the next outputs
    const uint16_t* r_x = A.x + ks * kFewK;
    const uint16_t* r_w = A.w + (int64_t)(beg / A.steps_k) * (NK ? (int64_t)kFewCols * A.K : kFewCols) + ks * step;
    auto request = [&](int stage) {
        const uint32_t to = lds0 + (uint32_t)(stage * kStage);
#pragma unroll
        for (int i = 0; i < kWCopies; ++i) copy_to_lds16(r_w, off_w[i], to + X::kBytes + (uint32_t)((i * 8 + wave) * 1024));
#pragma unroll
        for (int i = 0; i < kXCopies; ++i) copy_to_lds16(r_x, off_x[i], to + to_x[i]);
        if (r_left > 1) {                                                   // past the last step: that one again, never used
            --r_left;
            r_x += kFewK;
            r_w += step;
            if (++r_ks == A.steps_k) { r_ks = 0; r_x = A.x; r_w += wrap; }
        }
    };
    f32x16 acc[TB];
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) acc[tb] = f32x16{};
    float* part = A.part + (int64_t)group * 2 * (32 * TB * kFewCols);
    float* half = reinterpret_cast<float*>(lds + kStages * kStage) + wn * 32 * 32;
#pragma unroll
    for (int s = 0; s < kStages - 1; ++s) request(s);
    int stage = 0;
    for (int s = beg; s < end; ++s) {
        wait_older_copies_and_barrier<(kStages - 2) * (kXCopies + kWCopies)>();
        const uint32_t tile = lds0 + (uint32_t)(stage * kStage);
        const typename X::Lane in_x = X::in_tile(at_x, tile + (uint32_t)(wk * 1024));
        const typename W::Lane in_w = W::in_tile(at_w, tile + X::kBytes + (uint32_t)(NK ? wn * 4096 + wk * 1024 : wk * 8192 + wn * 1024));
        bf16x8 w[2], x[2][TB];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            w[t] = NK ? W::rows_operand(in_w, 0, 0, t) : W::cols_operand(in_w, 0, 16 * t, 0);
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) x[t][tb] = NK ? X::rows_operand(in_x, 0, 32 * tb, t) : X::rows_in_c_order(in_x, 32 * tb, t);
        }
        request(stage == 0 ? kStages - 1 : stage - 1);
        stage = stage + 1 == kStages ? 0 : stage + 1;
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) acc[tb] = mfma32(w[t], x[t][tb], acc[tb]);
        if (++ks == A.steps_k || s + 1 == end) {
            // the halves of the contraction meet in LDS, 32 rows at a time
            float* mine = half + (lane & 31) * 4 + h * 128;                 // [b][h][row][4]
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) {
                if (wk == 1) {
#pragma unroll
                    for (int b = 0; b < 4; ++b)
                        *reinterpret_cast<f32x4*>(mine + b * 256) = f32x4{acc[tb][4 * b], acc[tb][4 * b + 1], acc[tb][4 * b + 2], acc[tb][4 * b + 3]};
                }
                __syncthreads();
                if (wk == 0) {
#pragma unroll
                    for (int b = 0; b < 4; ++b) {
                        const f32x4 v = *reinterpret_cast<const f32x4*>(mine + b * 256);
                        *reinterpret_cast<f32x4*>(part + (32 * tb + (lane & 31)) * kFewCols + 32 * wn + 8 * b + 4 * h) =
                            f32x4{acc[tb][4 * b], acc[tb][4 * b + 1], acc[tb][4 * b + 2], acc[tb][4 * b + 3]} + v;
                    }
                }
                __syncthreads();
                acc[tb] = f32x16{};
            }
            part += 32 * TB * kFewCols;
            ks = 0;
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");                // stores and copies share a counter
        }
    }
}

// out = bf16(sum of the partial sums of its block, in the order of the contraction); a thread has 8 outputs of a row
__global__ __launch_bounds__(256) void few_rows_sum_kernel(const FewArgs A, int rows_part) {
    const int per_row = A.N / 8, i = blockIdx.x * 256 + threadIdx.x;
    if (i >= A.T * per_row) return;
    const int t = i / per_row, col = (i % per_row) * 8, block = col / kFewCols;
    const int first = few_group(A, block * A.steps_k), last = few_group(A, (block + 1) * A.steps_k - 1);
    const int64_t plane = (int64_t)rows_part * kFewCols;
    const float* p = A.part + t * kFewCols + col % kFewCols;
    auto slot = [&](int g) { return p + (2 * (int64_t)g + (g == first ? block - few_first(A, g) / A.steps_k : 0)) * plane; };
    f32x4 a = {}, b = {};
    for (int g = first; g <= last; g += 4) {
        f32x4 u[4], v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float* s = slot(min(g + j, last));
            u[j] = *reinterpret_cast<const f32x4*>(s);
            v[j] = *reinterpret_cast<const f32x4*>(s + 4);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (g + j <= last) { a += u[j]; b += v[j]; }
    }
    const float f[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    st16(A.out + (int64_t)t * A.N + col, pack8(f));
}

static int few_blocks(int64_t T) {                     // 32-row blocks the kernel is built for
    return (int)cdiv(T, 32);
}
static bool few_shape(int64_t T, int64_t N, int64_t K) {
    return T > 0 && T <= kFewMaxRows && N > 0 && K > 0 && N % kFewCols == 0 && K % kFewK == 0 && N * K < (int64_t)1 << 31;
}
static void few_steps(FewArgs& A) {
    const int blocks = A.N / kFewCols;
    A.steps_k = A.K / kFewK;
    A.total = blocks * A.steps_k;
    const int most = A.total / 4 < kFewUnits ? A.total / 4 : kFewUnits;    // four steps or more each: fewer do not pay for a start
    A.groups = most > blocks ? most : blocks;                              // at least a block's steps of a block: two partial sums at most
}

template <int TB>
static void few_launch(const FewArgs& A, bool nk, hipStream_t st) {
    if (nk) few_rows_kernel<TB, true><<<A.groups, 512, 0, st>>>(A);
    else few_rows_kernel<TB, false><<<A.groups, 512, 0, st>>>(A);
}

}  // namespace hyc

using namespace hyc;

extern "C" int64_t hyc_few_rows_workspace(int64_t T, int64_t N, int64_t K) {
    if (!few_shape(T, N, K)) return 0;
    FewArgs A = {};
    A.N = (int)N; A.K = (int)K;
    few_steps(A);
    return (int64_t)A.groups * 2 * 32 * few_blocks(T) * kFewCols * 4;
}

extern "C" int hyc_few_rows(const void* x, const void* w, int w_is_nk, void* out, void* workspace, int64_t workspace_bytes, int64_t T,
                            int64_t N, int64_t K, void* stream) {
    if (!few_shape(T, N, K)) return HYC_ERR_SHAPE;
    if (!x || !w || !out || !workspace) return HYC_ERR_NULL;
    if (!aligned16(x) || !aligned16(w) || !aligned16(out) || !aligned16(workspace)) return HYC_ERR_ALIGN;
    if (workspace_bytes < hyc_few_rows_workspace(T, N, K)) return HYC_ERR_WORKSPACE;
    FewArgs A = {};
    A.x = (const uint16_t*)x; A.w = (const uint16_t*)w; A.part = (float*)workspace; A.out = (uint16_t*)out;
    A.T = (int)T; A.N = (int)N; A.K = (int)K;
    few_steps(A);
    hipStream_t st = (hipStream_t)stream;
    const int tb = few_blocks(T);
    switch (tb) {
        case 1: few_launch<1>(A, w_is_nk != 0, st); break;
        case 2: few_launch<2>(A, w_is_nk != 0, st); break;
        case 3: few_launch<3>(A, w_is_nk != 0, st); break;
        default: few_launch<4>(A, w_is_nk != 0, st); break;
    }
    few_rows_sum_kernel<<<dim3((unsigned)cdiv(T * N / 8, 256)), 256, 0, st>>>(A, 32 * tb);
    return check_launch();
}
