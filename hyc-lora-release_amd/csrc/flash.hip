// Attention without a map, forward and backward, on the gfx950 matrix cores (causal or not, grouped key / value heads).
// q, o, grad_o, grad_q: bf16 [B, S, H, D]; k, v, grad_k, grad_v: bf16 [B, S, KV, D]; lse, delta: fp32 [B, H, S].
//
// Bound by the matrix cores and the vector units beside them (one exponential per score; 46 % and 60 % busy in the forward).
// A wave owns 32 rows of one axis (their operands stay in registers) and walks the other axis in tiles of 64 rows that its
// workgroup of four waves stages in LDS, double-buffered, copied asynchronously while the previous tile is worked on: two
// workgroups (128 KB) and two waves per SIMD are resident, one wave's exponentials beside the other's products.  Scores are
// formed transposed (a lane holds one row of the softmax), so the row sums need one exchange between the two halves of a wave
// and the probabilities are the next product's operand as they stand.  The backward runs as two kernels, one per owned axis,
// and forms scores twice instead of adding query gradients with atomics: the same bits on every run.
// [1, 8192, 32 heads, 128], causal, inside a layer step: forward 550 to 570 us (0.98 PFLOP/s), backward 700 + 920 to 740 + 980 us
// (1.15 PFLOP/s of its seven products, 0.82 counting five); the library kernels behind torch's scaled_dot_product_attention took
// 1280 and 5330.  The first version of
// the tile (rows of whole 256 bytes, addresses formed per read, every product waiting for the operand read right before it)
// took 615 and 2400 us.
#include "hyc_attn_tile.hpp"

namespace hyc {

constexpr int kFlashRows = 128;        // query (key) rows of a workgroup: 32 per wave
constexpr int kFlashTile = 64;         // rows of the tile the workgroup walks along the other axis

// Head of a workgroup: consecutive workgroups go to the 8 XCDs in turn, so heads that share keys and values (and all
// blocks of one head) are given numbers that meet on one XCD's L2.
__device__ __forceinline__ int head_of(int j, int heads) { return heads % 8 ? j : (j % 8) * (heads / 8) + j / 8; }

// whether a step has to look for masked entries: steps in the middle of a sequence are compiled without
template <bool B> struct Edge { static constexpr bool value = B; };

struct FlashArgs {
    const uint16_t *q, *k, *v, *o, *grad_o;
    uint16_t *out, *grad_q, *grad_k, *grad_v;
    float *lse, *delta;
    int B, S, H, KV;
    float scale;
};

template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 2) void flash_fwd_kernel(const FlashArgs A) {
    using Tile = AttnTile<D, kFlashTile>;
    constexpr int kOther = 2 * Tile::kBytes;                    // the second tensor's pair of tiles
    __shared__ __attribute__((aligned(1024))) char lds[4 * Tile::kBytes];       // two of keys, two of values
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int heads = A.B * A.H, nblk = (int)gridDim.x / heads;
    const int bh = head_of((int)blockIdx.x % heads, heads), blk = nblk - 1 - (int)blockIdx.x / heads;     // longest first
    const int b = bh / A.H, head = bh % A.H, kvh = head / (A.H / A.KV);
    const int ldq = A.H * D, ldk = A.KV * D;
    const uint16_t* kbase = A.k + ((int64_t)b * A.S * A.KV + kvh) * D;
    const uint16_t* vbase = A.v + ((int64_t)b * A.S * A.KV + kvh) * D;
    const int q0 = blk * kFlashRows + wave * 32, qrow = q0 + (lane & 31);
    const int qsafe = qrow < A.S ? qrow : A.S - 1;
    const float scale2 = A.scale * kLog2e;
    bf16x8 Q[D / 16];
    load_row_operands<D>(A.q + ((int64_t)b * A.S + qsafe) * ldq + head * D, h, Q);

    const int kend = CAUSAL ? min(A.S, blk * kFlashRows + kFlashRows) : A.S;
    const int tiles = (kend + kFlashTile - 1) / kFlashTile;
    const int full = CAUSAL ? blk * (kFlashRows / kFlashTile) : A.S / kFlashTile;    // tiles without an edge for any wave
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    const typename Tile::Lane at(lane);
    auto request = [&](int it) {
        Tile::request(kbase, it * kFlashTile, A.S - 1, ldk, lds0 + (it & 1) * Tile::kBytes, wave, lane);
        Tile::request(vbase, it * kFlashTile, A.S - 1, ldk, lds0 + (2 + (it & 1)) * Tile::kBytes, wave, lane);
    };
    request(0);

    f32x16 O[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) O[db] = f32x16{};
    float m = -INFINITY, l = 0.0f;
    auto step = [&](int it, auto edge) {
        const int k0 = it * kFlashTile;
        const typename Tile::Lane in = Tile::in_tile(at, lds0 + (it & 1) * Tile::kBytes);
        f32x16 s[2];
        s[0] = f32x16{}; s[1] = f32x16{};
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {
            s[0] = mfma32(Tile::rows_operand(in, 0, 0, t), Q[t], s[0]);
            s[1] = mfma32(Tile::rows_operand(in, 0, 32, t), Q[t], s[1]);
        }
        order_products<D / 8, 1, 6>();
        if (edge.value) {
            const int last = CAUSAL ? min(qrow, A.S - 1) : A.S - 1;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (k0 + 32 * kb + 8 * (r / 4) + 4 * h + r % 4 > last) s[kb][r] = -INFINITY;
        }
        float mx = s[0][0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[0][r]);
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[1][r]);
        mx = half_max(mx) * scale2;
        // The exact running maximum, so that a row's largest weight is 1 without rounding: letting the maximum lag (by up to
        // 2^8, which saves most of these multiplications) moved 41 % instead of 36 % of the outputs of 8192 keys off the
        // correctly rounded value.
        if (__any(mx > m)) {
            const float mn = fmaxf(m, mx), f = __builtin_amdgcn_exp2f(m - mn);
            m = mn;
            l *= f;
#pragma unroll
            for (int db = 0; db < D / 32; ++db)
#pragma unroll
                for (int r = 0; r < 16; ++r) O[db][r] *= f;
        }
        float sum = 0.0f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[kb][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][r], scale2, -m));
                sum += s[kb][r];
            }
        l += sum;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            const bf16x8 P = c_as_operand(s[t >> 1], t & 1);
#pragma unroll
            for (int db = 0; db < D / 32; ++db) O[db] = mfma32(Tile::cols_operand(in, kOther, 16 * t, 32 * db), P, O[db]);
        }
        order_products<D / 8, 2, 4>();
    };
    int it = 0;
    for (; it < full; ++it) {
        wait_copies_and_barrier();
        if (it + 1 < tiles) request(it + 1);
        step(it, Edge<false>{});
    }
    for (; it < tiles; ++it) {
        wait_copies_and_barrier();
        if (it + 1 < tiles) request(it + 1);
        if (!CAUSAL || it * kFlashTile <= q0 + 31) step(it, Edge<true>{});      // else nothing for this wave's rows; the barriers stay shared
    }
    l = half_sum(l);
    if (qrow < A.S) {
        store_rows<D>(A.out + ((int64_t)b * A.S + qrow) * ldq + head * D, h, O, 1.0f / l);
        if (h == 0) A.lse[((int64_t)b * A.H + head) * A.S + qrow] = (m + __builtin_amdgcn_logf(l)) * kLn2;
    }
}

// grad_q of 128 query rows; leaves -delta = -sum_d grad_o * o and the log-sum-exps to base 2 of these rows for the key /
// value kernel
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 2) void flash_bwd_q_kernel(const FlashArgs A) {
    using Tile = AttnTile<D, kFlashTile>;
    constexpr int kOther = 2 * Tile::kBytes;                    // the second tensor's pair of tiles
    __shared__ __attribute__((aligned(1024))) char lds[4 * Tile::kBytes];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int heads = A.B * A.H, nblk = (int)gridDim.x / heads;
    const int bh = head_of((int)blockIdx.x % heads, heads), blk = nblk - 1 - (int)blockIdx.x / heads;
    const int b = bh / A.H, head = bh % A.H, kvh = head / (A.H / A.KV);
    const int ldq = A.H * D, ldk = A.KV * D;
    const uint16_t* kbase = A.k + ((int64_t)b * A.S * A.KV + kvh) * D;
    const uint16_t* vbase = A.v + ((int64_t)b * A.S * A.KV + kvh) * D;
    const int q0 = blk * kFlashRows + wave * 32, qrow = q0 + (lane & 31);
    const int qsafe = qrow < A.S ? qrow : A.S - 1;
    const float scale2 = A.scale * kLog2e;
    const int64_t row_off = ((int64_t)b * A.S + qsafe) * ldq + head * D;
    bf16x8 Q[D / 16], G[D / 16];
    load_row_operands<D>(A.q + row_off, h, Q);
    load_row_operands<D>(A.grad_o + row_off, h, G);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    const typename Tile::Lane at(lane);
    auto request = [&](int it) {
        Tile::request(kbase, it * kFlashTile, A.S - 1, ldk, lds0 + (it & 1) * Tile::kBytes, wave, lane);
        Tile::request(vbase, it * kFlashTile, A.S - 1, ldk, lds0 + (2 + (it & 1)) * Tile::kBytes, wave, lane);
    };
    request(0);

    float delta = 0.0f;
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
        float a[8], g[8];
        unpack8(ld16(A.o + row_off + 16 * t + 8 * h), a);
        unpack8(__builtin_bit_cast(u32x4, G[t]), g);
#pragma unroll
        for (int j = 0; j < 8; ++j) delta = __builtin_fmaf(a[j], g[j], delta);
    }
    delta = half_sum(delta);
    const int64_t stat = ((int64_t)b * A.H + head) * A.S + qsafe;
    const float lse2 = A.lse[stat] * kLog2e;
    if (qrow < A.S && h == 0) {
        A.delta[stat] = -delta;
        A.delta[(int64_t)heads * A.S + stat] = lse2;
    }

    const int kend = CAUSAL ? min(A.S, blk * kFlashRows + kFlashRows) : A.S;
    const int tiles = (kend + kFlashTile - 1) / kFlashTile;
    const int full = CAUSAL ? blk * (kFlashRows / kFlashTile) : A.S / kFlashTile;
    f32x16 dq[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) dq[db] = f32x16{};
    auto step = [&](int it, auto edge) {
        const int k0 = it * kFlashTile;
        const typename Tile::Lane in = Tile::in_tile(at, lds0 + (it & 1) * Tile::kBytes);
        const int last = CAUSAL ? min(qrow, A.S - 1) : A.S - 1;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            f32x16 s = f32x16{}, dp = f32x16{};
#pragma unroll
            for (int t = 0; t < D / 16; ++t) {
                s = mfma32(Tile::rows_operand(in, 0, 32 * kb, t), Q[t], s);
                dp = mfma32(Tile::rows_operand(in, kOther, 32 * kb, t), G[t], dp);
            }
            order_products<D / 8, 1, 6>();
            if (edge.value) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (k0 + 32 * kb + 8 * (r / 4) + 4 * h + r % 4 > last) s[r] = -INFINITY;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r)
                s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], scale2, -lse2)) * (dp[r] - delta);
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const bf16x8 dS = c_as_operand(s, t);
#pragma unroll
                for (int db = 0; db < D / 32; ++db)
                    dq[db] = mfma32(Tile::cols_operand(in, 0, 32 * kb + 16 * t, 32 * db), dS, dq[db]);
            }
            order_products<D / 16, 2, 3>();
        }
    };
    int it = 0;
    for (; it < full; ++it) {
        wait_copies_and_barrier();
        if (it + 1 < tiles) request(it + 1);
        step(it, Edge<false>{});
    }
    for (; it < tiles; ++it) {
        wait_copies_and_barrier();
        if (it + 1 < tiles) request(it + 1);
        if (!CAUSAL || it * kFlashTile <= q0 + 31) step(it, Edge<true>{});
    }
    if (qrow < A.S) store_rows<D>(A.grad_q + row_off, h, dq, A.scale);
}

// grad_k and grad_v of 128 key rows of one key / value head, over all query rows of the head's group
template <int D, bool CAUSAL>
__global__ __launch_bounds__(256, 2) void flash_bwd_kv_kernel(const FlashArgs A) {
    using Tile = AttnTile<D, kFlashTile>;
    constexpr int kOther = 2 * Tile::kBytes;                    // the second tensor's pair of tiles
    constexpr int kStat = 256;                                  // bytes of 64 row statistics
    __shared__ __attribute__((aligned(1024))) char lds[4 * Tile::kBytes + 4 * kStat];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int heads = A.B * A.KV, group = A.H / A.KV;
    const int bh = head_of((int)blockIdx.x % heads, heads), blk = (int)blockIdx.x / heads;      // causal: block 0 is the longest
    const int b = bh / A.KV, kvh = bh % A.KV;
    const int ldq = A.H * D, ldk = A.KV * D;
    const int key0 = blk * kFlashRows + wave * 32, key = key0 + (lane & 31);
    const int ksafe = key < A.S ? key : A.S - 1;
    const float scale2 = A.scale * kLog2e;
    const int64_t row_off = ((int64_t)b * A.S + ksafe) * ldk + kvh * D;
    bf16x8 K[D / 16], V[D / 16];
    load_row_operands<D>(A.k + row_off, h, K);
    load_row_operands<D>(A.v + row_off, h, V);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    const typename Tile::Lane at(lane);
    const int first = CAUSAL ? blk * kFlashRows / kFlashTile : 0;             // first query tile that sees these keys
    const int per_head = (A.S + kFlashTile - 1) / kFlashTile - first;
    const int tiles = per_head * group;
    const uint16_t* qb = A.q + (int64_t)b * A.S * ldq + kvh * group * D;
    const uint16_t* gb = A.grad_o + (int64_t)b * A.S * ldq + kvh * group * D;
    const float* delta_b = A.delta + ((int64_t)b * A.H + kvh * group) * A.S;
    const float* lse_b = delta_b + (int64_t)A.B * A.H * A.S;

    auto request = [&](int g, int q0, int buf) {
        Tile::request(qb + g * D, q0, A.S - 1, ldq, lds0 + buf * Tile::kBytes, wave, lane);
        Tile::request(gb + g * D, q0, A.S - 1, ldq, lds0 + (2 + buf) * Tile::kBytes, wave, lane);
        const uint32_t row = (uint32_t)(q0 + lane < A.S ? q0 + lane : A.S - 1) * 4u;
        if (wave == 0) copy_to_lds4(lse_b + (int64_t)g * A.S, row, lds0 + 4 * Tile::kBytes + buf * kStat);
        if (wave == 1) copy_to_lds4(delta_b + (int64_t)g * A.S, row, lds0 + 4 * Tile::kBytes + (2 + buf) * kStat);
    };
    request(0, first * kFlashTile, 0);
    f32x16 dk[D / 32], dv[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) dk[db] = dv[db] = f32x16{};
    auto step = [&](int q0, int buf, bool edge) {
        const typename Tile::Lane in = Tile::in_tile(at, lds0 + buf * Tile::kBytes);
        const uint32_t stat = lds0 + 4 * Tile::kBytes + buf * kStat + 16 * h;
        typedef const __attribute__((address_space(3))) f32x4 lds_f32x4;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            f32x16 s = f32x16{}, dp;
#pragma unroll
            for (int b4 = 0; b4 < 4; ++b4) {                    // grad_o v^T - delta: the sums start from -delta
                const f32x4 del = *(lds_f32x4*)(stat + 2 * kStat + (32 * half + 8 * b4) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) dp[4 * b4 + e] = del[e];
            }
#pragma unroll
            for (int t = 0; t < D / 16; ++t) {
                s = mfma32(Tile::rows_operand(in, 0, 32 * half, t), K[t], s);
                dp = mfma32(Tile::rows_operand(in, kOther, 32 * half, t), V[t], dp);
            }
#pragma unroll
            for (int b4 = 0; b4 < 4; ++b4) {
                const f32x4 lse = *(lds_f32x4*)(stat + (32 * half + 8 * b4) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int r = 4 * b4 + e;
                    s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], scale2, -lse[e]));
                    dp[r] = s[r] * dp[r];
                }
            }
            if (edge) {
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int row = q0 + 32 * half + 8 * (r / 4) + 4 * h + r % 4;
                    if (row >= A.S || (CAUSAL && row < key)) s[r] = dp[r] = 0.0f;
                }
            }
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const bf16x8 P = c_as_operand(s, t), dS = c_as_operand(dp, t);
#pragma unroll
                for (int db = 0; db < D / 32; ++db) {
                    dv[db] = mfma32(Tile::cols_operand(in, kOther, 32 * half + 16 * t, 32 * db), P, dv[db]);
                    dk[db] = mfma32(Tile::cols_operand(in, 0, 32 * half + 16 * t, 32 * db), dS, dk[db]);
                }
            }
            order_products<D / 8, 2, 3>();
        }
    };
    int g = 0, tile = 0;                                        // the tile being worked on
    for (int it = 0; it < tiles; ++it) {
        wait_copies_and_barrier();
        const int q0 = (first + tile) * kFlashTile, buf = it & 1;
        if (++tile == per_head) { tile = 0; ++g; }
        if (it + 1 < tiles) request(g, (first + tile) * kFlashTile, buf ^ 1);
        if (CAUSAL && q0 + kFlashTile - 1 < key0) continue;    // nothing for this wave's keys; the barriers stay shared
        step(q0, buf, (CAUSAL && q0 < key0 + 31) || q0 + kFlashTile > A.S);
    }
    if (key < A.S) {
        store_rows<D>(A.grad_k + row_off, h, dk, A.scale);
        store_rows<D>(A.grad_v + row_off, h, dv, 1.0f);
    }
}

int flash_check(int64_t B, int64_t S, int64_t H, int64_t KV, int64_t D) {
    if (B < 0 || S < 0 || H <= 0 || KV <= 0 || H % KV || (D != 64 && D != 128)) return HYC_ERR_SHAPE;
    if (S > (1 << 20) || S * H * D > (int64_t)1 << 30) return HYC_ERR_SHAPE;                                        // 32-bit offsets inside a batch element
    if (B * H > 1 << 23 || cdiv(S, kFlashRows) * B * H > 1 << 23) return HYC_ERR_SHAPE;                             // fewer than 2^32 threads a launch
    return HYC_OK;
}

}  // namespace hyc

using namespace hyc;

extern "C" int hyc_flash_fwd(const void* q, const void* k, const void* v, void* o, float* lse, int64_t B, int64_t S, int64_t H,
                             int64_t KV, int64_t D, float scale, int causal, void* stream) {
    const int rc = flash_check(B, S, H, KV, D);
    if (rc != HYC_OK) return rc;
    if (B == 0 || S == 0) return HYC_OK;
    if (!q || !k || !v || !o || !lse) return HYC_ERR_NULL;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o)) return HYC_ERR_ALIGN;
    FlashArgs A = {};
    A.q = (const uint16_t*)q; A.k = (const uint16_t*)k; A.v = (const uint16_t*)v; A.out = (uint16_t*)o; A.lse = lse;
    A.B = (int)B; A.S = (int)S; A.H = (int)H; A.KV = (int)KV; A.scale = scale;
    const dim3 grid((unsigned)(cdiv(S, kFlashRows) * B * H));
    hipStream_t st = (hipStream_t)stream;
    if (D == 128) { if (causal) flash_fwd_kernel<128, true><<<grid, 256, 0, st>>>(A); else flash_fwd_kernel<128, false><<<grid, 256, 0, st>>>(A); }
    else { if (causal) flash_fwd_kernel<64, true><<<grid, 256, 0, st>>>(A); else flash_fwd_kernel<64, false><<<grid, 256, 0, st>>>(A); }
    return check_launch();
}

extern "C" int hyc_flash_bwd(const void* grad_o, const void* q, const void* k, const void* v, const void* o, const float* lse,
                             float* delta, void* grad_q, void* grad_k, void* grad_v, int64_t B, int64_t S, int64_t H, int64_t KV,
                             int64_t D, float scale, int causal, void* stream) {
    const int rc = flash_check(B, S, H, KV, D);
    if (rc != HYC_OK) return rc;
    if (B == 0 || S == 0) return HYC_OK;
    if (!grad_o || !q || !k || !v || !o || !lse || !delta || !grad_q || !grad_k || !grad_v) return HYC_ERR_NULL;
    for (const void* p : {grad_o, q, k, v, o, (const void*)grad_q, (const void*)grad_k, (const void*)grad_v})
        if (!aligned16(p)) return HYC_ERR_ALIGN;
    FlashArgs A = {};
    A.q = (const uint16_t*)q; A.k = (const uint16_t*)k; A.v = (const uint16_t*)v; A.o = (const uint16_t*)o; A.grad_o = (const uint16_t*)grad_o;
    A.grad_q = (uint16_t*)grad_q; A.grad_k = (uint16_t*)grad_k; A.grad_v = (uint16_t*)grad_v; A.lse = const_cast<float*>(lse); A.delta = delta;
    A.B = (int)B; A.S = (int)S; A.H = (int)H; A.KV = (int)KV; A.scale = scale;
    const dim3 gq((unsigned)(cdiv(S, kFlashRows) * B * H)), gkv((unsigned)(cdiv(S, kFlashRows) * B * KV));
    hipStream_t st = (hipStream_t)stream;
#define HYC_FLASH_BWD(DD, CC) do { flash_bwd_q_kernel<DD, CC><<<gq, 256, 0, st>>>(A); flash_bwd_kv_kernel<DD, CC><<<gkv, 256, 0, st>>>(A); } while (0)
    if (D == 128) { if (causal) HYC_FLASH_BWD(128, true); else HYC_FLASH_BWD(128, false); }
    else { if (causal) HYC_FLASH_BWD(64, true); else HYC_FLASH_BWD(64, false); }
#undef HYC_FLASH_BWD
    return check_launch();
}
