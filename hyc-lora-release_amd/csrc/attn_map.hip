// Attention through a softmax map that is kept sparse, on the gfx950 matrix cores: scores, softmax, the kept entries and the
// attention output without a dense map in memory, and the backward straight from the kept entries.
//
//   t = bf16(bf16(bf16(q k^T) * scale) + mask),  p = bf16(softmax_fp32(t)),  o = p v            (forward)
//   g = bf16(grad_o v^T),  d = sum_row bf16(a * g),  ds = bf16(bf16((g - d) * a) * scale)       (backward; a: the kept p)
//   grad_q = ds k,  grad_k = ds^T q,  grad_v = a^T grad_o
// with the roundings the separate kernels have (softmax_map.hip), so that a map made here is the map they would make from
// the same scores.  q, o: bf16 [B, S, H, D]; k, v: bf16 [B, S, KV, D].
//
// Bound by the vector units (roundings, two exponentials per score and walk) with the matrix cores beside them; the tiles and
// the division of a workgroup are those of flash.hip.  Per element the dense route moved 2 bytes nine times (scores, map,
// kept entries, restored map, both gradients); here only the entries move.  [4, 1024, 32 heads, 128], causal, 5 % kept:
// forward 106 us and entries 80 us (library products, softmax with count, compaction: 357 us), backward 237 us (products,
// restore + softmax backward: 537 us).  Of these, 6 and 14 us are the looks at the operands for NaN and infinities.
#include "hyc_attn_tile.hpp"

namespace hyc {

constexpr int kMapRows = 128;          // query (key) rows of a workgroup: 32 per wave
constexpr int kMapTile = 64;           // keys of a tile
constexpr int kMapMax = 4096;          // longest row: 64 tiles, one bit each
constexpr float kDead = -1e30f;        // a mask entry at or below takes its key out of the softmax
constexpr int kSegElems = 4096;        // elements of a segment of the compressed map

struct MapArgs {
    const uint16_t *q, *k, *v, *mask;
    int64_t mask_sb, mask_sr;          // element strides of the mask's batches and rows (0: shared)
    uint16_t *o, *map;                 // map: dense copy, or NULL
    const float* threshold;            // NULL: nothing is counted
    float *row_max, *row_inv;          // per row of the map
    uint32_t *counts, *block_counts;   // kept entries of a row; of the 32 rows of a wave
    const uint64_t* classes;           // per mask batch and 32 rows: tiles with a live entry, tiles without a mask entry but 0
    const uint32_t* wild;              // per key / value head 64 words, a byte per 16 rows of a tile: not 0 if one is not finite
    uint32_t* walked_all;              // per workgroup of the forward: whether it walked every tile after all
    const int64_t* row_offsets;
    int64_t *indices, *seg_offsets;
    uint16_t* values;
    int64_t capacity;
    int B, S, H, KV;
    float scale;
};

// 16 rows of a tile of keys and of values, looked at by one wave: is an element infinite or NaN?
template <int D>
__device__ __forceinline__ bool tile_is_wild(const uint16_t* k, const uint16_t* v, int ld, int row0, int row_last, int lane) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    constexpr int kLanes = D / 8, kRows = 64 / kLanes, kLoads = 16 / kRows;      // lanes of a row, rows of a load
    u32x4 e[2 * kLoads];
#pragma unroll
    for (int i = 0; i < kLoads; ++i) {
        const int64_t at = (int64_t)min(row0 + i * kRows + lane / kLanes, row_last) * ld + lane % kLanes * 8;
        e[2 * i] = ld16(k + at);
        e[2 * i + 1] = ld16(v + at);
    }
    u16x2 most = {0, 0};
#pragma unroll
    for (int i = 0; i < 2 * kLoads; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, e[i][j] & 0x7fff7fffu));
    return __any(most.x >= 0x7f80 || most.y >= 0x7f80);
}

// Which tiles matter.  Of the mask: bit t of classes[..][0] is set when some entry of the 32 rows x 64 keys is above kDead, of
// classes[..][1] when all are zero.  A wave looks at 8 tiles (a byte of either word), a lane at 8 keys of the 32 rows; a
// causal mask lets half of the tiles go.  Of the keys and values: tiles may only go where all of a head's are finite, since a
// weight of 0 times an infinite value, or an infinite score under a mask of -inf, is NaN (one read of both, 6 us of 106 at
// [4, 1024, 32 heads, 128]).
template <int D>
__global__ __launch_bounds__(256) void map_classes_kernel(const MapArgs A, int mask_wgs, int mask_batches) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, S = A.S, bytes = (S + 511) / 512, blocks = (S + 31) / 32;
    if ((int)blockIdx.x >= mask_wgs * mask_batches) {
        const int i = (int)blockIdx.x - mask_wgs * mask_batches, nt = (S + kMapTile - 1) / kMapTile;
        const int kvh = i % A.KV, t = i / A.KV % nt, b = i / A.KV / nt;
        const int64_t at = ((int64_t)b * S * A.KV + kvh) * D;
        const bool w = tile_is_wild<D>(A.k + at, A.v + at, A.KV * D, t * kMapTile + wave * 16, S - 1, lane);
        if (lane == 0) reinterpret_cast<uint8_t*>(const_cast<uint32_t*>(A.wild))[((int64_t)(b * A.KV + kvh) * 64 + t) * 4 + wave] = w;
        return;
    }
    const int mb = (int)blockIdx.x / mask_wgs, unit = (int)blockIdx.x % mask_wgs * 4 + wave;
    if (unit >= blocks * bytes) return;
    const int rb = unit / bytes, step = unit % bytes, key = step * 512 + lane * 8;
    const int64_t sr = A.mask_sr;
    const uint16_t* base = A.mask + (int64_t)mb * A.mask_sb + (int64_t)rb * 32 * sr;
    const int rows = sr == 0 ? 1 : min(32, S - rb * 32);
    bool any = false, zero = true;
    if (key < S) {
        for (int r0 = 0; r0 < rows; r0 += 8) {
            u32x4 v[8];
#pragma unroll
            for (int i = 0; i < 8; ++i) v[i] = ld16(base + (int64_t)min(r0 + i, rows - 1) * sr + key);
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                float f[8];
                unpack8(v[i], f);
#pragma unroll
                for (int j = 0; j < 8; ++j) { any |= !(f[j] <= kDead); zero &= f[j] == 0.0f; }
            }
        }
    }
    const uint64_t a = __ballot(any), z = __ballot(!zero);
    uint32_t live = 0, plain = 0;
#pragma unroll
    for (int t = 0; t < 8; ++t) {
        if ((a >> (8 * t)) & 0xff) live |= 1u << t;
        if (!((z >> (8 * t)) & 0xff)) plain |= 1u << t;
    }
    if (lane == 0) {
        uint8_t* out = reinterpret_cast<uint8_t*>(const_cast<uint64_t*>(A.classes)) + ((int64_t)mb * blocks + rb) * 16 + step;
        out[0] = (uint8_t)live;
        out[8] = (uint8_t)plain;
    }
}

// A float p rounds to a bf16 value above `thr` (and not to zero) exactly when !(p <= keep_limit(thr)); NaN is kept.
__device__ __forceinline__ float keep_limit(float thr) {
    const uint32_t b = __builtin_bit_cast(uint32_t, rbf(thr));
    if ((b & 0x7f800000u) == 0x7f800000u && !(b & 0x80000000u)) return INFINITY;
    if (b & 0x80000000u) return (b & 0x7fffffffu) > 0x7f800000u ? INFINITY : __builtin_bit_cast(float, 0x8000u);
    return __builtin_bit_cast(float, b + ((b & 0x10000u) ? 0x7fffu : 0x8000u));
}

// blocks of 32 rows that the waves of a head's workgroups own (the last ones may lie past its rows)
__host__ __device__ inline int64_t row_blocks(int64_t S) { return (S + kMapRows - 1) / kMapRows * (kMapRows / 32); }

__device__ __forceinline__ uint64_t tiles_of(int S) {
    const int n = (S + kMapTile - 1) / kMapTile;
    return n >= 64 ? ~0ull : (1ull << n) - 1;
}

__device__ __forceinline__ uint64_t uniform64(uint64_t v) {
    return (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(v >> 32)) << 32 | (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
// keeps the compiler from moving a wave's LDS accesses across; the hardware does them in order
__device__ __forceinline__ void lds_order() { asm volatile("" ::: "memory"); }

// What a wave knows about its 32 rows
struct MapRows {
    int b, head, kvh, q0, qrow, row_in;          // row_in: qrow, or the last row
    int64_t flat;                                // row of the map [B * H * S]
    uint64_t live, plain, wg_live;               // tiles of the wave; tiles any wave of the workgroup needs
    const uint16_t* mrow;
};

template <int D>
__device__ __forceinline__ MapRows map_rows(const MapArgs& A, int lane, int wave) {
    MapRows R;
    const int heads = A.B * A.H, nblk = (int)gridDim.x / heads;
    const int j = (int)blockIdx.x % heads, blk = nblk - 1 - (int)blockIdx.x / heads;
    const int bh = heads % 8 ? j : (j % 8) * (heads / 8) + j / 8;            // heads that share keys on one XCD
    R.b = bh / A.H; R.head = bh % A.H; R.kvh = R.head / (A.H / A.KV);
    R.q0 = blk * kMapRows + wave * 32;
    R.qrow = R.q0 + (lane & 31);
    R.row_in = R.qrow < A.S ? R.qrow : A.S - 1;
    R.flat = (int64_t)bh * A.S + R.row_in;
    const uint64_t all = tiles_of(A.S);
    R.live = R.plain = R.wg_live = all;
    R.mrow = nullptr;
    if (A.mask) {
        const int nrb = (A.S + 31) / 32;
        const uint64_t* c = A.classes + (int64_t)(A.mask_sb ? R.b : 0) * nrb * 2;
        const int own = min(R.q0 / 32, nrb - 1);
        R.live = uniform64(c[2 * own] & all);
        R.plain = uniform64(c[2 * own + 1]);
        R.wg_live = 0;
        for (int w = 0; w < 4; ++w) R.wg_live |= c[2 * min(blk * 4 + w, nrb - 1)] & all;
        R.wg_live = uniform64(R.wg_live);
        const uint32_t* w = A.wild + (int64_t)(R.b * A.KV + R.kvh) * 64;
        if (__any(lane < (A.S + kMapTile - 1) / kMapTile && w[lane] != 0)) R.live = R.wg_live = all;
        R.mrow = A.mask + (int64_t)R.b * A.mask_sb + (int64_t)R.row_in * A.mask_sr;
    }
    return R;
}

// t of 64 keys: s[kb][r] belongs to key k0 + 32*kb + 8*(r/4) + 4h + r%4; keys past the row give -inf
template <int D, class Tile>
__device__ __forceinline__ void map_scores(const MapArgs& A, const MapRows& R, const typename Tile::Lane& in, const bf16x8 (&Q)[D / 16], int k0,
                                           bool plain, int h, f32x16 (&s)[2]) {
    u32x2 mv[8];
    if (!plain) {
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const int key = k0 + 8 * b + 4 * h;
            mv[b] = u32x2{0, 0};
            if (key < A.S) mv[b] = ld8(R.mrow + key);
        }
    }
    s[0] = f32x16{}; s[1] = f32x16{};
#pragma unroll
    for (int t = 0; t < D / 16; ++t) {
        s[0] = mfma32(Tile::rows_operand(in, 0, 0, t), Q[t], s[0]);
        s[1] = mfma32(Tile::rows_operand(in, 0, 32, t), Q[t], s[1]);
    }
    order_products<D / 8, 1, 6>();
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = rbf(rbf(s[kb][r]) * A.scale);
    if (!plain) {
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint32_t lo = mv[b].x, hi = mv[b].y;
            f32x16& c = s[b >> 2];
            const int r = 4 * (b & 3);
            c[r] = rbf(c[r] + bf_lo(lo)); c[r + 1] = rbf(c[r + 1] + bf_hi(lo));
            c[r + 2] = rbf(c[r + 2] + bf_lo(hi)); c[r + 3] = rbf(c[r + 3] + bf_hi(hi));
        }
    }
    if (k0 + kMapTile > A.S) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (k0 + 32 * kb + 8 * (r / 4) + 4 * h + r % 4 >= A.S) s[kb][r] = -INFINITY;
    }
}

// Walks the tiles of `todo` with the copies of the next one in flight.  `buf`: the buffer to fill next; body(tile, buffer).
template <class Request, class Body>
__device__ __forceinline__ void walk_tiles(uint64_t todo, int& buf, Request request, Body body) {
    if (!todo) return;
    int cur = __builtin_ctzll(todo);
    request(cur, buf);
    while (todo) {
        wait_copies_and_barrier();
        todo &= todo - 1;
        const int next = todo ? __builtin_ctzll(todo) : 0;
        if (todo) request(next, buf ^ 1);
        body(cur, buf);
        cur = next;
        buf ^= 1;
    }
}

__device__ __forceinline__ float prob(float t, float m, float inv) { return __builtin_amdgcn_exp2f((t - m) * kLog2e) * inv; }

// Probabilities of a tile's 64 keys, in place.  Keys past the row get 0, whatever the row's sum is: in a row of NaN scores or of
// nothing but -inf, `inv` is not finite and prob(-inf) is NaN, which counts as kept.
__device__ __forceinline__ void map_probs(const MapArgs& A, int k0, int h, float m, float inv, f32x16 (&s)[2]) {
#pragma unroll
    for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = prob(s[kb][r], m, inv);
    if (k0 + kMapTile > A.S) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (k0 + 32 * kb + 8 * (r / 4) + 4 * h + r % 4 >= A.S) s[kb][r] = 0.0f;
    }
}

// Row maxima and sums in a first walk over the keys, the probabilities, their count and the output in a second: a
// probability is rounded to bf16 relative to its row's final sum, so an online softmax cannot form it.
template <int D>
__global__ __launch_bounds__(256, 2) void map_fwd_kernel(const MapArgs A) {
    using Tile = AttnTile<D, kMapTile>;
    constexpr int kOther = 2 * Tile::kBytes;
    __shared__ __attribute__((aligned(1024))) char lds[4 * Tile::kBytes];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    MapRows R = map_rows<D>(A, lane, wave);
    const int ldq = A.H * D, ldk = A.KV * D;
    const uint16_t* kbase = A.k + ((int64_t)R.b * A.S * A.KV + R.kvh) * D;
    const uint16_t* vbase = A.v + ((int64_t)R.b * A.S * A.KV + R.kvh) * D;
    bf16x8 Q[D / 16];
    load_row_operands<D>(A.q + ((int64_t)R.b * A.S + R.row_in) * ldq + R.head * D, h, Q);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    const typename Tile::Lane at(lane);
    int buf = 0;
    auto request_k = [&](int t, int b) { Tile::request(kbase, t * kMapTile, A.S - 1, ldk, lds0 + b * Tile::kBytes, wave, lane); };
    auto request_kv = [&](int t, int b) {
        request_k(t, b);
        Tile::request(vbase, t * kMapTile, A.S - 1, ldk, lds0 + (2 + b) * Tile::kBytes, wave, lane);
    };
    float m = -INFINITY, l = 0.0f;
    for (int attempt = 0; attempt < 2; ++attempt) {
        walk_tiles(R.wg_live, buf, request_k, [&](int t, int b) {
            if (!((R.live >> t) & 1)) return;
            f32x16 s[2];
            map_scores<D, Tile>(A, R, Tile::in_tile(at, lds0 + b * Tile::kBytes), Q, t * kMapTile, (R.plain >> t) & 1, h, s);
            float mx = s[0][0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[0][r]);
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[1][r]);
            const float mn = fmaxf(m, half_max(mx));
            const float ms = mn == -INFINITY ? 0.0f : mn;
            float sum = 0.0f;
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
#pragma unroll
                for (int r = 0; r < 16; ++r) sum += __builtin_amdgcn_exp2f((s[kb][r] - ms) * kLog2e);
            l = l * __builtin_amdgcn_exp2f((m - ms) * kLog2e) + sum;
            m = mn;
        });
        // A row none of whose live tiles holds a live entry of its own (a padded query: all its keys are masked) needs the
        // entries that were left out: with a finite mask value they all weigh the same.  So does a row whose sum is NaN: its
        // weights are NaN at every key.
        if (attempt == 1 || !A.mask) break;
        const bool again = __syncthreads_or(m <= 0.5f * kDead || l != l);
        if (A.threshold && threadIdx.x == 0) A.walked_all[blockIdx.x] = again;
        if (!again) break;
        R.live = R.wg_live = tiles_of(A.S);
        m = -INFINITY;
        l = 0.0f;
    }
    l = half_sum(l);
    const float row_max = m;
    if (m == -INFINITY) m = 0.0f;
    const float inv = 1.0f / l;
    float limit = INFINITY;
    if (A.threshold) limit = keep_limit(*A.threshold);

    f32x16 O[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) O[db] = f32x16{};
    uint32_t count = 0;
    uint16_t* mrow = A.map ? A.map + R.flat * A.S : nullptr;
    walk_tiles(mrow ? tiles_of(A.S) : R.wg_live, buf, request_kv, [&](int t, int b) {
        const int k0 = t * kMapTile;
        const bool live = (R.live >> t) & 1;
        if (!live) {
            if (mrow && R.qrow < A.S) {
#pragma unroll
                for (int i = 0; i < 8; ++i)
                    if (k0 + 8 * i + 4 * h < A.S) st8(mrow + k0 + 8 * i + 4 * h, u32x2{0, 0});
            }
            return;
        }
        f32x16 s[2];
        const typename Tile::Lane in = Tile::in_tile(at, lds0 + b * Tile::kBytes);
        map_scores<D, Tile>(A, R, in, Q, k0, (R.plain >> t) & 1, h, s);
        map_probs(A, k0, h, m, inv, s);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (!(s[kb][r] <= limit)) ++count;
        bf16x8 P[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) P[i] = c_as_operand(s[i >> 1], i & 1);
        if (mrow && R.qrow < A.S) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                const u32x4 w = __builtin_bit_cast(u32x4, P[i >> 1]);
                const u32x2 v = (i & 1) ? u32x2{w.z, w.w} : u32x2{w.x, w.y};
                if (k0 + 8 * i + 4 * h < A.S) st8(mrow + k0 + 8 * i + 4 * h, v);
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int db = 0; db < D / 32; ++db) O[db] = mfma32(Tile::cols_operand(in, kOther, 16 * i, 32 * db), P[i], O[db]);
        order_products<D / 8, 2, 4>();
    });
    if (R.qrow < A.S) store_rows<D>(A.o + ((int64_t)R.b * A.S + R.qrow) * ldq + R.head * D, h, O, 1.0f);
    if (A.threshold) {
        const u32x2 both = __builtin_amdgcn_permlane32_swap(count, count, false, false);
        const uint32_t kept = R.qrow < A.S ? both.x + both.y : 0u;
        if (R.qrow < A.S && h == 0) {
            A.row_max[R.flat] = row_max;
            A.row_inv[R.flat] = inv;
            A.counts[R.flat] = kept;
        }
        const uint32_t up_to = wave_inclusive_scan(kept);
        if (lane == 31) A.block_counts[(int64_t)(R.b * A.H + R.head) * row_blocks(A.S) + R.q0 / 32] = up_to;
    }
}

// row_offsets[r] = kept entries of the rows before r, for every r up to B * H * S.  A workgroup scans the 1024 counts of its own
// rows and adds up what lies before them by itself, from the counts of 32 rows: these reads grow with the square of the rows.
// Forward with the count, [2048, 128, 16 heads, 64]: 675 us (573 without it); from the counts of single rows 1911.
__global__ __launch_bounds__(1024) void map_row_scan_kernel(const uint32_t* counts, const uint32_t* block_counts, int64_t rows, int S, int64_t* offsets) {
    __shared__ long long front_part[16];
    __shared__ uint32_t wave_total[16];
    const int t = threadIdx.x, lane = t & (kWave - 1), wave = t >> 6;
    const int64_t base = (int64_t)blockIdx.x * 1024, blocks = base / S * row_blocks(S) + base % S / 32;
    long long front = t < (int)(base % S % 32) ? counts[base - 1 - t] : 0;
    for (int64_t f = t; f < blocks; f += 4 * 1024) {
        uint32_t v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = f + u * 1024 < blocks ? block_counts[f + u * 1024] : 0u;
#pragma unroll
        for (int u = 0; u < 4; ++u) front += v[u];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) front += __shfl_xor(front, o, kWave);
    const int64_t row = base + t;
    const uint32_t c = row < rows ? counts[row] : 0u, inc = wave_inclusive_scan(c);
    if (lane == 0) front_part[wave] = front;
    if (lane == kWave - 1) wave_total[wave] = inc;
    __syncthreads();
    long long at = 0;
    uint32_t before = 0, total = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
        at += front_part[w];
        before += w < wave ? wave_total[w] : 0u;
        total += wave_total[w];
    }
    if (row < rows) offsets[row] = at + before + (inc - c);
    if (t == 0 && base + 1024 >= rows) offsets[rows] = at + total;
}

// A 32-row x 64-key bf16 tile that one wave keeps in LDS: rows of 128 bytes, their 16-byte chunks permuted by the row.
struct MapPatch {
    static constexpr int kBytes = 32 * 128;
    __device__ static __forceinline__ uint32_t at(int row, int key) { return (uint32_t)(row * 128 + (((key >> 3) ^ (row & 7)) << 4) + (key & 7) * 2); }
};

// The kept entries, in the order of the flattened map: scores and probabilities once more (the same instructions, the same
// bits), each row's entries behind those of the rows before it.
template <int D>
__global__ __launch_bounds__(256, 2) void map_emit_kernel(const MapArgs A) {
    using Tile = AttnTile<D, kMapTile>;
    __shared__ __attribute__((aligned(1024))) char lds[2 * Tile::kBytes + 4 * MapPatch::kBytes];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    MapRows R = map_rows<D>(A, lane, wave);
    const int ldq = A.H * D, ldk = A.KV * D;
    const uint16_t* kbase = A.k + ((int64_t)R.b * A.S * A.KV + R.kvh) * D;
    bf16x8 Q[D / 16];
    load_row_operands<D>(A.q + ((int64_t)R.b * A.S + R.row_in) * ldq + R.head * D, h, Q);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    const typename Tile::Lane at(lane);
    char* patch = lds + 2 * Tile::kBytes + wave * MapPatch::kBytes;
    const float row_max = A.row_max[R.flat], m = row_max == -INFINITY ? 0.0f : row_max;
    const float inv = A.row_inv[R.flat], limit = keep_limit(*A.threshold);
    const bool valid = R.qrow < A.S;
    if (A.mask && A.walked_all[blockIdx.x]) R.live = R.wg_live = tiles_of(A.S);
    int64_t at_out = A.row_offsets[R.flat];
    const int64_t elem0 = R.flat * A.S;
    const int64_t total = A.row_offsets[(int64_t)A.B * A.H * A.S];
    const int64_t elems = (int64_t)A.B * A.H * A.S * A.S;
    if (blockIdx.x == 0 && threadIdx.x == 0) A.seg_offsets[(elems + kSegElems - 1) / kSegElems] = total;
    int buf = 0, done = 0;                                          // tiles of the row whose segment starts have been written
    // segment starts in [k0, k1) of the row, with `bits` the kept keys of the 64 from k0 on
    auto segments = [&](int k0, int k1, uint64_t bits) {
        if (!valid || h != 0) return;
        for (int64_t e = (elem0 + k0 + kSegElems - 1) / kSegElems * kSegElems; e < elem0 + k1; e += kSegElems)
            A.seg_offsets[e / kSegElems] = at_out + __popcll(bits & ((1ull << (uint32_t)(e - elem0 - k0)) - 1));
    };
    walk_tiles(R.wg_live, buf, [&](int t, int b) { Tile::request(kbase, t * kMapTile, A.S - 1, ldk, lds0 + b * Tile::kBytes, wave, lane); },
               [&](int t, int b) {
        if (!((R.live >> t) & 1)) return;
        const int k0 = t * kMapTile;
        f32x16 s[2];
        map_scores<D, Tile>(A, R, Tile::in_tile(at, lds0 + b * Tile::kBytes), Q, k0, (R.plain >> t) & 1, h, s);
        map_probs(A, k0, h, m, inv, s);
        uint32_t own[2] = {0, 0};
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int r = 0; r < 16; ++r) own[kb] |= !(s[kb][r] <= limit) ? 1u << (8 * (r / 4) + r % 4) : 0u;
        uint32_t full[2];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            const uint32_t w = valid ? own[kb] << (4 * h) : 0u;
            const u32x2 both = __builtin_amdgcn_permlane32_swap(w, w, false, false);
            full[kb] = both.x | both.y;
        }
        const uint64_t bits = (uint64_t)full[1] << 32 | full[0];
        if (done < t) segments(done * kMapTile, k0, 0);             // tiles in between keep nothing
        segments(k0, min(k0 + kMapTile, A.S), bits);
        done = t + 1;
        if (__any(bits != 0)) {
#pragma unroll
            for (int b8 = 0; b8 < 8; ++b8) {
                const f32x16& c = s[b8 >> 2];
                const int r = 4 * (b8 & 3);
                *reinterpret_cast<u32x2*>(patch + MapPatch::at(lane & 31, 8 * b8 + 4 * h)) = u32x2{pk_bf16(c[r], c[r + 1]), pk_bf16(c[r + 2], c[r + 3])};
            }
            lds_order();
            uint32_t w = h ? full[1] : full[0];
            int64_t pos = at_out + (h ? __popc(full[0]) : 0);
            while (__any(w != 0)) {
                if (w) {
                    const int key = 32 * h + __builtin_ctz(w);
                    w &= w - 1;
                    if (pos < A.capacity) {
                        A.indices[pos] = elem0 + k0 + key;
                        A.values[pos] = *reinterpret_cast<const uint16_t*>(patch + MapPatch::at(lane & 31, key));
                    }
                    ++pos;
                }
            }
            lds_order();
            at_out += __popcll(bits);
        }
    });
    segments(done * kMapTile, A.S, 0);
}

// ---- backward ---------------------------------------------------------------------------------------------------------
struct MapBwdArgs {
    const uint16_t *grad_o, *q, *k, *v;
    const int64_t *indices, *seg_offsets;
    const uint16_t* values;
    uint32_t* entries;                  // (row % 32 * 64 + key % 64) << 16 | value, grouped by 32-row x 64-key tile
    uint16_t* grads;                    // per entry: the map's gradient, then the score's
    uint32_t* tile_at;                  // [B * H * row blocks, tiles + 1]: where a tile's entries begin
    uint32_t* wild;                     // [B * H * row blocks]: what of the 32 rows is not finite, kWildQ | ...
    uint32_t* wild_columns;             // [B * H * row blocks][3][4]: columns of q, k and grad_o that hold such an element, where wild says so
    uint16_t *grad_q, *grad_k, *grad_v;
    int B, S, H, KV;
    float scale;
};

// Groups the entries of 32 rows by tile of 64 keys.  The entries of a tile come in no particular order (each has its own
// place in the dense tile that the kernels below rebuild from them, so no result depends on it).
__global__ __launch_bounds__(256) void map_regroup_kernel(const MapBwdArgs A) {
    __shared__ uint32_t place[kMapMax / kMapTile], below[2];
    const int nrb = (A.S + 31) / 32, nt = (A.S + kMapTile - 1) / kMapTile;
    const int bh = blockIdx.x / nrb, r0 = (int)(blockIdx.x % nrb) * 32;
    const int64_t elems = (int64_t)A.B * A.H * A.S * A.S;
    const int64_t e0 = ((int64_t)bh * A.S + r0) * A.S, e1 = e0 + (int64_t)min(32, A.S - r0) * A.S;
    if (threadIdx.x < (unsigned)nt) place[threadIdx.x] = 0;
    if (threadIdx.x < 2) below[threadIdx.x] = 0;
    __syncthreads();
    int64_t edge[2];
#pragma unroll
    for (int s = 0; s < 2; ++s) {                               // first entry at or past e0 (e1): in the segment that holds it
        const int64_t e = s ? e1 : e0;
        edge[s] = A.seg_offsets[e < elems ? e / kSegElems : (elems + kSegElems - 1) / kSegElems];
        if (e < elems && e % kSegElems) {
            const int64_t end = A.seg_offsets[e / kSegElems + 1];
            uint32_t n = 0;
            for (int64_t i = edge[s] + threadIdx.x; i < end; i += 256) n += A.indices[i] < e;
            if (n) atomicAdd(&below[s], n);
        }
    }
    __syncthreads();
    const int64_t first = edge[0] + below[0], last = edge[1] + below[1];
    const float inv = 1.0f / (float)A.S;
    auto split = [&](uint32_t rel, uint32_t& row, uint32_t& key) {           // rel < 32 * 4096: exact in fp32, off by one at most
        row = (uint32_t)((float)rel * inv);
        if (row * (uint32_t)A.S > rel) --row;
        if ((row + 1) * (uint32_t)A.S <= rel) ++row;
        key = rel - row * (uint32_t)A.S;
    };
    for (int64_t i = first + threadIdx.x; i < last; i += 256) {
        uint32_t row, key;
        split((uint32_t)(A.indices[i] - e0), row, key);
        atomicAdd(&place[key / kMapTile], 1u);
    }
    __syncthreads();
    if (threadIdx.x < 64) {
        const uint32_t n = (int)threadIdx.x < nt ? place[threadIdx.x] : 0u;
        const uint32_t at = (uint32_t)first + wave_inclusive_scan(n) - n;
        uint32_t* out = A.tile_at + (int64_t)blockIdx.x * (nt + 1);
        if ((int)threadIdx.x < nt) out[threadIdx.x] = place[threadIdx.x] = at;
        if (threadIdx.x == 0) out[nt] = (uint32_t)last;
    }
    __syncthreads();
    for (int64_t i = first + threadIdx.x; i < last; i += 256) {
        uint32_t row, key;
        split((uint32_t)(A.indices[i] - e0), row, key);
        const uint32_t slot = atomicAdd(&place[key / kMapTile], 1u);
        A.entries[slot] = (row * kMapTile + key % kMapTile) << 16 | A.values[i];
    }
}

// Entries of a tile that a wave holds in registers: 64 of each of kHeld loads.  With 5 % of a causal map kept, the tiles below
// the diagonal hold 200 on average; the few fuller ones (a row's first keys) are worked through kHeld loads at a time.
constexpr int kHeld = 4;

// Entries that are not kept are never formed, but they are 0 only while everything is finite: 0 times an infinite value, or an
// infinite gradient of the map times their 0, is NaN.  What follows, for one head of the formulas on top:
//   grad_o[i, c] not finite:  d_i, so row i of grad_q and all of grad_k; column c of grad_v
//   v not finite:             every d, so all of grad_q and grad_k
//   d_i not finite (an entry that is NaN):  row i of grad_q, all of grad_k
//   k[j, c] not finite:       column c of grad_q
//   q[i, c] not finite:       column c of grad_k
// The kernel of grad_q looks at the rows of its numbers in all four and sees to the rows; the kernel of grad_k and grad_v, which
// runs after it, sees to the columns and to the rest.  The looks are one read of the operands: 14 us of 237 at [4, 1024, 32
// heads, 128], 8 of 280 at [1, 2048, 32, 128] (14 and 17 in the kernel that groups the entries, where nothing else of theirs is read).
enum : uint32_t { kWildQ = 1, kWildK = 2, kWildV = 4, kWildG = 8, kWildD = 16 };

// Elements of 16 bytes that are infinite or NaN: is there one, and which (bit j: element j)?
template <int N>
__device__ __forceinline__ bool any_wild(const u32x4 (&e)[N]) {
    typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
    u16x2 most = {0, 0};
#pragma unroll
    for (int i = 0; i < N; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) most = __builtin_elementwise_max(most, __builtin_bit_cast(u16x2, e[i][j] & 0x7fff7fffu));
    return most.x >= 0x7f80 || most.y >= 0x7f80;
}
__device__ __forceinline__ uint32_t wild_bits(u32x4 e) {
    uint32_t m = 0;
#pragma unroll
    for (int j = 0; j < 8; ++j) m |= ((e[j / 2] >> (16 * (j & 1))) & 0x7f80u) == 0x7f80u ? 1u << j : 0u;
    return m;
}
// 32 rows of a tensor as a wave reads them fastest, whole rows side by side: lane l has chunk l % (D / 8) of every (512 / D)th row
template <int D>
struct WildRows {
    static constexpr int kLanes = D / 8, kLoads = 32 * kLanes / 64;
    u32x4 e[kLoads];
    __device__ __forceinline__ void request(const uint16_t* base, int64_t ld, int row0, int row_last, int lane) {
#pragma unroll
        for (int i = 0; i < kLoads; ++i) e[i] = ld16(base + (int64_t)min(row0 + (i * 64 + lane) / kLanes, row_last) * ld + lane % kLanes * 8);
    }
    // the columns with such an element, a bit each, as D / 8 bytes
    __device__ __forceinline__ void note_columns(uint8_t* out, int lane) const {
        uint32_t m = 0;
#pragma unroll
        for (int i = 0; i < kLoads; ++i) m |= wild_bits(e[i]);
#pragma unroll
        for (int o = kLanes; o < 64; o *= 2) m |= (uint32_t)__shfl_xor((int)m, o, kWave);
        if (lane < kLanes) out[lane] = (uint8_t)m;
    }
};

// Clears a wave's 32 x 64 patch
__device__ __forceinline__ void clear_patch(char* patch, int lane) {
#pragma unroll
    for (int i = 0; i < 4; ++i) *reinterpret_cast<u32x4*>(patch + i * 1024 + lane * 16) = u32x4{0, 0, 0, 0};
}

// grad_q of 128 rows.  First walk: g at the kept entries and the row sums d (the tile of a is rebuilt in LDS, the products of
// one tile are 32 x 64 values of which a few percent are kept).  Second walk: ds from g, d and a per entry, its tile rebuilt in
// LDS as the operand of ds k; ds stays in `grads` for the key / value kernel.  Tiles without an entry are left out.
template <int D>
__global__ __launch_bounds__(256, 2) void map_bwd_q_kernel(const MapBwdArgs A) {
    using Tile = AttnTile<D, kMapTile>;
    __shared__ __attribute__((aligned(1024))) char lds[2 * Tile::kBytes + 4 * MapPatch::kBytes + 4 * 128 + 32];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int heads = A.B * A.H, nblk = (int)gridDim.x / heads, nrb = (A.S + 31) / 32, nt = (A.S + kMapTile - 1) / kMapTile;
    const int j = (int)blockIdx.x % heads, blk = nblk - 1 - (int)blockIdx.x / heads;
    const int bh = heads % 8 ? j : (j % 8) * (heads / 8) + j / 8;
    const int b = bh / A.H, head = bh % A.H, kvh = head / (A.H / A.KV);
    const int ldq = A.H * D, ldk = A.KV * D;
    const int rb = blk * 4 + wave, qrow = rb * 32 + (lane & 31), row_in = qrow < A.S ? qrow : A.S - 1;
    const uint16_t* kbase = A.k + ((int64_t)b * A.S * A.KV + kvh) * D;
    const uint16_t* vbase = A.v + ((int64_t)b * A.S * A.KV + kvh) * D;
    const int64_t row_off = ((int64_t)b * A.S + row_in) * ldq + head * D;
    bf16x8 G[D / 16];
    load_row_operands<D>(A.grad_o + row_off, h, G);
    WildRows<D> q_rows, k_rows, v_rows;                                 // looked at below, while the first tile is on its way
    const bool lead = head % (A.H / A.KV) == 0;                         // a group's keys and values: looked at by its first head
    q_rows.request(A.q + ((int64_t)b * A.S * A.H + head) * D, ldq, rb * 32, A.S - 1, lane);
    if (lead) {
        k_rows.request(kbase, ldk, rb * 32, A.S - 1, lane);
        v_rows.request(vbase, ldk, rb * 32, A.S - 1, lane);
    }
    char* patch = lds + 2 * Tile::kBytes + wave * MapPatch::kBytes;
    float* row_sum = reinterpret_cast<float*>(lds + 2 * Tile::kBytes + 4 * MapPatch::kBytes + wave * 128);
    uint64_t* wave_tiles = reinterpret_cast<uint64_t*>(lds + 2 * Tile::kBytes + 4 * MapPatch::kBytes + 4 * 128);
    const uint32_t* tile_at = A.tile_at + ((int64_t)bh * nrb + min(rb, nrb - 1)) * (nt + 1);
    const uint32_t t_beg = rb < nrb ? tile_at[min(lane, nt)] : 0u, t_end = rb < nrb ? tile_at[min(lane + 1, nt)] : 0u;     // of tile `lane`
    const uint64_t own = __ballot(lane < nt && t_end > t_beg);
    if (lane == 0) wave_tiles[wave] = own;
    __syncthreads();
    const uint64_t todo = uniform64(wave_tiles[0] | wave_tiles[1] | wave_tiles[2] | wave_tiles[3]);
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    const typename Tile::Lane at(lane);
    // The entries of a tile (the first 64 * kHeld; more are read when they are used) are requested one tile ahead: their loads and
    // the copies of the next tile come back in the order they were issued, so a use right after the request would wait for all.
    uint32_t beg = 0, n = 0, e[kHeld] = {}, gr[kHeld] = {};
    auto load = [&](uint32_t from, bool with_grads) {                   // entries from .. of the tile (past its end: the last again)
#pragma unroll
        for (int i = 0; i < kHeld; ++i) {
            const uint32_t k = beg + min(from + (uint32_t)(lane + 64 * i), n - 1);
            e[i] = A.entries[k];
            if (with_grads) gr[i] = A.grads[k];
        }
    };
    auto fetch = [&](uint64_t tiles, bool with_grads) {
        n = 0;
        if (!tiles) return;
        const int t = __builtin_ctzll(tiles);
        beg = (uint32_t)__builtin_amdgcn_readlane((int)t_beg, t);
        n = (uint32_t)__builtin_amdgcn_readlane((int)t_end, t) - beg;
        load(0, with_grads);
    };
    auto later = [&](int t) { return t < 63 ? own >> (t + 1) << (t + 1) : 0ull; };
    int buf = 0;
    float d = 0.0f;
    fetch(own, false);
    uint32_t marks = 0;                                                 // of the wave's rows
    {
        uint8_t* columns = reinterpret_cast<uint8_t*>(A.wild_columns + ((int64_t)bh * nrb + min(rb, nrb - 1)) * 12);
        if (__any(any_wild(q_rows.e))) {
            marks |= kWildQ;
            if (rb < nrb) q_rows.note_columns(columns, lane);
        }
        if (lead) {
            if (__any(any_wild(k_rows.e))) {
                marks |= kWildK;
                if (rb < nrb) k_rows.note_columns(columns + 16, lane);
            }
            if (__any(any_wild(v_rows.e))) marks |= kWildV;
        }
    }
    u32x4 g_rows[D / 16];
#pragma unroll
    for (int t = 0; t < D / 16; ++t) g_rows[t] = __builtin_bit_cast(u32x4, G[t]);
    const bool wild_g = any_wild(g_rows);
    if (__any(wild_g)) {
        marks |= kWildG;
        uint8_t* columns = reinterpret_cast<uint8_t*>(A.wild_columns + ((int64_t)bh * nrb + min(rb, nrb - 1)) * 12 + 8);
#pragma unroll
        for (int t = 0; t < D / 16; ++t) {                              // lane l: columns 16t + 8h .. of row l % 32
            uint32_t m = wild_bits(g_rows[t]);
#pragma unroll
            for (int o = 1; o < 32; o *= 2) m |= (uint32_t)__shfl_xor((int)m, o, kWave);
            if (rb < nrb && (lane & 31) == 0) columns[2 * t + h] = (uint8_t)m;
        }
    }
    walk_tiles(todo, buf, [&](int t, int bb) { Tile::request(vbase, t * kMapTile, A.S - 1, ldk, lds0 + bb * Tile::kBytes, wave, lane); },
               [&](int t, int bb) {
        if (!((own >> t) & 1)) return;
        clear_patch(patch, lane);
        const typename Tile::Lane in = Tile::in_tile(at, lds0 + bb * Tile::kBytes);
        f32x16 g[2];
        g[0] = f32x16{}; g[1] = f32x16{};
#pragma unroll
        for (int i = 0; i < D / 16; ++i) {
            g[0] = mfma32(Tile::rows_operand(in, 0, 0, i), G[i], g[0]);
            g[1] = mfma32(Tile::rows_operand(in, 0, 32, i), G[i], g[1]);
        }
        order_products<D / 8, 1, 6>();
        lds_order();
        auto put = [&](uint32_t v) { *reinterpret_cast<uint16_t*>(patch + MapPatch::at(v >> 22, (v >> 16) & 63)) = (uint16_t)v; };
        for (uint32_t from = 0;;) {
#pragma unroll
            for (int i = 0; i < kHeld; ++i) if (from + (uint32_t)(lane + 64 * i) < n) put(e[i]);
            from += 64 * kHeld;
            if (from >= n) break;
            load(from, false);
        }
        lds_order();
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            u32x2* at8 = reinterpret_cast<u32x2*>(patch + MapPatch::at(lane & 31, 8 * i + 4 * h));
            const u32x2 a = *at8;
            const uint32_t a0 = a.x, a1 = a.y;
            const f32x16& c = g[i >> 2];
            const int r = 4 * (i & 3);
            const uint32_t g0 = pk_bf16(c[r], c[r + 1]), g1 = pk_bf16(c[r + 2], c[r + 3]);
            d += rbf(bf_lo(a0) * bf_lo(g0));
            d += rbf(bf_hi(a0) * bf_hi(g0));
            d += rbf(bf_lo(a1) * bf_lo(g1));
            d += rbf(bf_hi(a1) * bf_hi(g1));
            *at8 = u32x2{g0, g1};
        }
        lds_order();
        auto get = [&](uint32_t v) { return *reinterpret_cast<const uint16_t*>(patch + MapPatch::at(v >> 22, (v >> 16) & 63)); };
        if (n > 64 * kHeld) load(0, false);
        for (uint32_t from = 0;;) {
#pragma unroll
            for (int i = 0; i < kHeld; ++i) if (from + (uint32_t)(lane + 64 * i) < n) A.grads[beg + from + lane + 64 * i] = get(e[i]);
            from += 64 * kHeld;
            if (from >= n) break;
            load(from, false);
        }
        lds_order();
        fetch(later(t), false);
    });
    if (wild_g) d = NAN;
    d = half_sum(d);
    if (lane < 32) row_sum[lane] = d;
    lds_order();
    const bool wild_row = !(__builtin_fabsf(d) < INFINITY);
    if (rb < nrb) {
        if (__any(wild_row)) marks |= kWildD;
        if (lane == 0) A.wild[(int64_t)bh * nrb + rb] = marks;
    }
    f32x16 dq[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) dq[db] = f32x16{};
    fetch(own, true);
    walk_tiles(todo, buf, [&](int t, int bb) { Tile::request(kbase, t * kMapTile, A.S - 1, ldk, lds0 + bb * Tile::kBytes, wave, lane); },
               [&](int t, int bb) {
        if (!((own >> t) & 1)) return;
        clear_patch(patch, lane);
        lds_order();
        auto put = [&](uint32_t i, uint32_t v, uint32_t g) {
            const uint16_t ds = f_to_bf(rbf((bf_to_f((uint16_t)g) - row_sum[v >> 22]) * bf_lo(v)) * A.scale);
            A.grads[beg + i] = ds;
            *reinterpret_cast<uint16_t*>(patch + MapPatch::at(v >> 22, (v >> 16) & 63)) = ds;
        };
        for (uint32_t from = 0;;) {
#pragma unroll
            for (int i = 0; i < kHeld; ++i) if (from + (uint32_t)(lane + 64 * i) < n) put(from + lane + 64 * i, e[i], gr[i]);
            from += 64 * kHeld;
            if (from >= n) break;
            load(from, true);
        }
        lds_order();
        fetch(later(t), true);
        const typename Tile::Lane in = Tile::in_tile(at, lds0 + bb * Tile::kBytes);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const u32x2 lo = *reinterpret_cast<const u32x2*>(patch + MapPatch::at(lane & 31, 16 * i + 4 * h));
            const u32x2 hi = *reinterpret_cast<const u32x2*>(patch + MapPatch::at(lane & 31, 16 * i + 8 + 4 * h));
            const bf16x8 dS = as_bf16x8(u32x4{lo.x, lo.y, hi.x, hi.y});
#pragma unroll
            for (int db = 0; db < D / 32; ++db) dq[db] = mfma32(Tile::cols_operand(in, 0, 16 * i, 32 * db), dS, dq[db]);
        }
        order_products<D / 8, 2, 4>();
        lds_order();
    });
    if (qrow < A.S) store_rows<D>(A.grad_q + row_off, h, dq, wild_row ? NAN : 1.0f);
}

// Rows row0 .. row0 + 31 of the three gradients of a head with something that is not finite: NaN over what has been stored
// there, in the columns that have it.  A lane overwrites what it stored itself (grad_k, grad_v) or what the kernel before left.
template <int D>
__device__ __forceinline__ void map_spread(const MapBwdArgs& A, int bh, int nrb, int row0, int lane, uint32_t marks) {
    const int h = lane >> 5, b = bh / A.H, head = bh % A.H, lead = bh - head % (A.H / A.KV), row = row0 + (lane & 31);
    const bool all_k = __any(marks & (kWildV | kWildD)), all_q = __any(marks & kWildV);
    const int64_t off = (((int64_t)b * A.S + row) * A.H + head) * D;
#pragma unroll 1
    for (int i = 0; i < D / 32; ++i) {
        uint32_t q = 0, k = 0, g = 0;
#pragma unroll 1
        for (int rb = 0; rb < nrb; ++rb) {
            const uint32_t own = A.wild[(int64_t)bh * nrb + rb], keys = A.wild[(int64_t)lead * nrb + rb];
            if (own & kWildQ) q |= A.wild_columns[((int64_t)bh * nrb + rb) * 12 + i];
            if (keys & kWildK) k |= A.wild_columns[((int64_t)lead * nrb + rb) * 12 + 4 + i];
            if (own & kWildG) g |= A.wild_columns[((int64_t)bh * nrb + rb) * 12 + 8 + i];
        }
        if (row >= A.S) continue;
#pragma unroll 1
        for (int c = 0; c < 32; ++c) {
            if (((c >> 2) & 1) != h) continue;
            if (all_k || (q >> c & 1)) A.grad_k[off + 32 * i + c] = 0x7fc0;
            if (g >> c & 1) A.grad_v[off + 32 * i + c] = 0x7fc0;
            if (all_q || (k >> c & 1)) A.grad_q[off + 32 * i + c] = 0x7fc0;
        }
    }
}

// grad_k and grad_v of 128 keys of one query head, over the rows that keep an entry there, 32 rows at a time: the transposed
// tiles of a and ds are rebuilt in LDS while the step before is worked on.  Grouped heads each give their own gradient, rounded
// (as the reference's copies of a key / value head do), and are added up afterwards: a workgroup per key / value head had to
// walk all rows of its group, with a quarter of the workgroups (583 us against 256 us on 32 heads over 8, [2, 2048]).
template <int D>
__global__ __launch_bounds__(256, 2) void map_bwd_kv_kernel(const MapBwdArgs A) {
    using Tile = AttnTile<D, 32>;
    constexpr int kOther = 2 * Tile::kBytes, kPatch = 64 * 64;          // 64 keys x 32 rows
    constexpr int kSteps = kMapMax / 32;
    __shared__ __attribute__((aligned(1024))) char lds[4 * Tile::kBytes + 8 * kPatch + kSteps * 12 + 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), h = lane >> 5;
    const int heads = A.B * A.H, nrb = (A.S + 31) / 32, nt = (A.S + kMapTile - 1) / kMapTile;
    const int j = (int)blockIdx.x % heads, blk = (int)blockIdx.x / heads;
    const int bh = heads % 8 ? j : (j % 8) * (heads / 8) + j / 8;
    const int b = bh / A.H, head = bh % A.H;
    const int ldq = A.H * D;
    const int key = blk * kMapRows + wave * 32 + (lane & 31);
    const int t0 = blk * 2, t1 = min(t0 + 1, nt), t2 = min(t0 + 2, nt);
    uint32_t marks = 0;                                                 // of the head; row blocks are at most 128
    {
        const int lead = bh - head % (A.H / A.KV);
        for (int i = 0; i < 2; ++i) {
            const int64_t rb = min(lane + 64 * i, nrb - 1);
            marks |= (A.wild[(int64_t)bh * nrb + rb] & ~(uint32_t)(kWildK | kWildV)) | (A.wild[(int64_t)lead * nrb + rb] & (kWildK | kWildV));
        }
    }
    const uint32_t* tile_at = A.tile_at + (int64_t)bh * nrb * (nt + 1);
    // a step: 32 rows with entries, where those of the first tile begin, how many they and the second's are
    uint32_t* steps = reinterpret_cast<uint32_t*>(lds + 4 * Tile::kBytes + 8 * kPatch);
    uint32_t* wave_n = steps + 3 * kSteps;
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_addr(lds));
    const typename Tile::Lane at(lane);
    const uint16_t* qb = A.q + (int64_t)b * A.S * ldq + head * D;
    const uint16_t* gb = A.grad_o + (int64_t)b * A.S * ldq + head * D;
    // wave w rebuilds tile w % 2 of the two, of a (w < 2) or of ds
    struct Pending { uint32_t beg, n, e[kHeld], v[kHeld]; };
    auto load = [&](Pending& p, uint32_t from) {
#pragma unroll
        for (int u = 0; u < kHeld; ++u) {
            const uint32_t k = from + (uint32_t)(lane + 64 * u);
            p.e[u] = p.v[u] = 0;
            if (k < p.n) {
                p.e[u] = A.entries[p.beg + k];
                if (wave >> 1) p.v[u] = A.grads[p.beg + k];
            }
        }
    };
    auto fetch = [&](int i) {                                           // the first entries of a tile, requested a step ahead
        Pending p;
        const uint32_t first = steps[3 * i + 1], both = steps[3 * i + 2];
        p.beg = __builtin_amdgcn_readfirstlane(wave & 1 ? first + (both & 0xffffu) : first);
        p.n = __builtin_amdgcn_readfirstlane(wave & 1 ? both >> 16 : both & 0xffffu);
        load(p, 0);
        return p;
    };
    auto rebuild = [&](Pending& p, int buf) {
        char* patch = lds + 4 * Tile::kBytes + (buf * 4 + wave) * kPatch;
        clear_patch(patch, lane);
        lds_order();
        auto put = [&](uint32_t e, uint32_t v) {
            const uint32_t row = e >> 22, k = (e >> 16) & 63;
            *reinterpret_cast<uint16_t*>(patch + k * 64 + (((row >> 3) ^ ((k >> 2) & 3)) << 4) + (row & 7) * 2) = (uint16_t)v;
        };
        for (uint32_t from = 0;;) {
#pragma unroll
            for (int u = 0; u < kHeld; ++u) if (from + (uint32_t)(lane + 64 * u) < p.n) put(p.e[u], wave >> 1 ? p.v[u] : p.e[u]);
            from += 64 * kHeld;
            if (from >= p.n) break;
            load(p, from);
        }
        lds_order();
    };
    auto request = [&](int i, int buf) {
        const int r0 = __builtin_amdgcn_readfirstlane((int)steps[3 * i]) * 32;
        Tile::request(qb, r0, A.S - 1, ldq, lds0 + buf * Tile::kBytes, wave, lane);
        Tile::request(gb, r0, A.S - 1, ldq, lds0 + (2 + buf) * Tile::kBytes, wave, lane);
    };
    f32x16 dk[D / 32], dv[D / 32];
#pragma unroll
    for (int db = 0; db < D / 32; ++db) dk[db] = dv[db] = f32x16{};
    int nsteps;
    {                                                                   // the steps in order: at most 128, one per thread of two waves
        const int s = threadIdx.x;
        uint32_t a0 = 0, a1 = 0, a2 = 0;
        if (s < nrb) {
            const uint32_t* r = tile_at + (int64_t)s * (nt + 1);
            a0 = r[t0]; a1 = r[t1]; a2 = r[t2];
        }
        const uint64_t m = __ballot(a2 > a0);
        if (lane == 0) wave_n[wave] = __popcll(m);
        __syncthreads();
        nsteps = wave_n[0] + wave_n[1];
        if (a2 > a0) {
            const int place = (wave ? wave_n[0] : 0) + __popcll(m & ((1ull << lane) - 1));
            steps[3 * place] = s;
            steps[3 * place + 1] = a0;
            steps[3 * place + 2] = (a1 - a0) | (a2 - a1) << 16;
        }
        __syncthreads();
    }
    nsteps = __builtin_amdgcn_readfirstlane(nsteps);
    Pending p = {};
    if (nsteps > 0) {
        request(0, 0);
        p = fetch(0);
        rebuild(p, 0);
        if (nsteps > 1) p = fetch(1);
    }
    for (int i = 0; i < nsteps; ++i) {
        const int buf = i & 1;
        wait_copies_and_barrier();
        if (i + 1 < nsteps) {
            request(i + 1, buf ^ 1);
            rebuild(p, buf ^ 1);
            if (i + 2 < nsteps) p = fetch(i + 2);
        }
        const typename Tile::Lane in = Tile::in_tile(at, lds0 + buf * Tile::kBytes);
        const int k = (wave & 1) * 32 + (lane & 31);
        const char* pa = lds + 4 * Tile::kBytes + (buf * 4 + (wave >> 1)) * kPatch + k * 64 + 8 * h;
        const char* pd = pa + 2 * kPatch;
        const int x = (k >> 2) & 3;
#pragma unroll
        for (int t = 0; t < 2; ++t) {
            const u32x2 a0 = *reinterpret_cast<const u32x2*>(pa + (((2 * t) ^ x) << 4)), a1 = *reinterpret_cast<const u32x2*>(pa + (((2 * t + 1) ^ x) << 4));
            const u32x2 d0 = *reinterpret_cast<const u32x2*>(pd + (((2 * t) ^ x) << 4)), d1 = *reinterpret_cast<const u32x2*>(pd + (((2 * t + 1) ^ x) << 4));
            const bf16x8 P = as_bf16x8(u32x4{a0.x, a0.y, a1.x, a1.y}), dS = as_bf16x8(u32x4{d0.x, d0.y, d1.x, d1.y});
#pragma unroll
            for (int db = 0; db < D / 32; ++db) {
                dv[db] = mfma32(Tile::cols_operand(in, kOther, 16 * t, 32 * db), P, dv[db]);
                dk[db] = mfma32(Tile::cols_operand(in, 0, 16 * t, 32 * db), dS, dk[db]);
            }
        }
        lds_order();
    }
    if (key < A.S) {
        const int64_t off = ((int64_t)b * A.S + key) * ldq + head * D;
        store_rows<D>(A.grad_k + off, h, dk, 1.0f);
        store_rows<D>(A.grad_v + off, h, dv, 1.0f);
    }
    if (__any(marks != 0)) map_spread<D>(A, bh, nrb, blk * kMapRows + wave * 32, lane, marks);
}

// out[t, kv, :] = sum of in[t, kv * group + 0 .. group - 1, :], fp32 sums in that order, one rounding; D / 8 chunks a row
__global__ __launch_bounds__(256) void group_sum_kernel(const uint16_t* __restrict__ in0, const uint16_t* __restrict__ in1, uint16_t* __restrict__ out0,
                                                        uint16_t* __restrict__ out1, int64_t chunks, int per_head, int group) {
    const int64_t c = blockIdx.x * 256ll + threadIdx.x;
    if (c >= chunks) return;
    const uint16_t* in = (blockIdx.y ? in1 : in0) + ((c / per_head) * group * per_head + c % per_head) * 8;
    float acc[8] = {};
    for (int g = 0; g < group; ++g) {
        float f[8];
        unpack8(ld16_nt(in + (int64_t)g * per_head * 8), f);
#pragma unroll
        for (int i = 0; i < 8; ++i) acc[i] += f[i];
    }
    st16((blockIdx.y ? out1 : out0) + c * 8, pack8(acc));
}

struct MapBwdWorkspace { int64_t entries, grads, tile_at, wild, wild_columns, heads, bytes; };
static MapBwdWorkspace map_bwd_workspace(int64_t B, int64_t S, int64_t H, int64_t KV, int64_t D, int64_t capacity) {
    auto up = [](int64_t v) { return cdiv(v, 256) * 256; };
    MapBwdWorkspace w;
    w.entries = 0;
    w.grads = up(capacity * 4);
    w.tile_at = w.grads + up(capacity * 2);
    w.wild = w.tile_at + up(B * H * cdiv(S, 32) * (cdiv(S, kMapTile) + 1) * 4);
    w.wild_columns = w.wild + up(B * H * cdiv(S, 32) * 4);
    w.heads = w.wild_columns + up(B * H * cdiv(S, 32) * 48);                             // per query head: grad_k, then grad_v
    w.bytes = w.heads + (H == KV ? 0 : 2 * up(B * S * H * D * 2));
    return w;
}

struct MapWorkspace {                   // offsets in bytes
    int64_t row_max, row_inv, counts, block_counts, row_offsets, classes, wild, walked_all, bytes;
};
static MapWorkspace map_workspace(int64_t B, int64_t S, int64_t H) {
    const int64_t rows = B * H * S, nrb = cdiv(S, 32);
    auto up = [](int64_t v) { return cdiv(v, 256) * 256; };
    MapWorkspace w;
    w.row_max = 0;
    w.row_inv = up(rows * 4);
    w.counts = w.row_inv + up(rows * 4);
    w.block_counts = w.counts + up(rows * 4);
    w.row_offsets = w.block_counts + up(B * H * row_blocks(S) * 4);
    w.classes = w.row_offsets + up((rows + 1) * 8);
    w.wild = w.classes + up(B * nrb * 16);
    w.walked_all = w.wild + up(B * H * 64 * 4);
    w.bytes = w.walked_all + up(cdiv(S, kMapRows) * B * H * 4);
    return w;
}

static int map_check(int64_t B, int64_t S, int64_t H, int64_t KV, int64_t D) {
    if (B < 0 || S < 0 || H <= 0 || KV <= 0 || H % KV || (D != 64 && D != 128) || S % 8 || S > kMapMax) return HYC_ERR_SHAPE;
    if (S * H * D > (int64_t)1 << 30 || B * H > 1 << 22 || cdiv(S, 32) * B * H > 1 << 22) return HYC_ERR_SHAPE;     // fewer than 2^32 threads a launch
    return HYC_OK;
}

}  // namespace hyc

using namespace hyc;

extern "C" int64_t hyc_map_workspace(int64_t B, int64_t S, int64_t H) { return B < 0 || S < 0 || H < 0 ? 0 : map_workspace(B, S, H).bytes; }

static MapArgs map_args(const void* q, const void* k, const void* mask, int64_t msb, int64_t msr, const float* threshold, void* workspace,
                        int64_t B, int64_t S, int64_t H, int64_t KV, float scale) {
    const MapWorkspace w = map_workspace(B, S, H);
    char* ws = (char*)workspace;
    MapArgs A = {};
    A.q = (const uint16_t*)q; A.k = (const uint16_t*)k; A.mask = (const uint16_t*)mask; A.mask_sb = msb; A.mask_sr = msr;
    A.threshold = threshold;
    A.row_max = (float*)(ws + w.row_max); A.row_inv = (float*)(ws + w.row_inv); A.counts = (uint32_t*)(ws + w.counts);
    A.block_counts = (uint32_t*)(ws + w.block_counts);
    A.row_offsets = (const int64_t*)(ws + w.row_offsets); A.classes = (const uint64_t*)(ws + w.classes);
    A.wild = (const uint32_t*)(ws + w.wild); A.walked_all = (uint32_t*)(ws + w.walked_all);
    A.B = (int)B; A.S = (int)S; A.H = (int)H; A.KV = (int)KV; A.scale = scale;
    return A;
}

extern "C" int hyc_map_fwd(const void* q, const void* k, const void* v, const void* mask, int64_t mask_stride_b, int64_t mask_stride_row,
                           void* o, void* map, const float* threshold, void* workspace, int64_t workspace_bytes, int64_t B, int64_t S,
                           int64_t H, int64_t KV, int64_t D, float scale, void* stream) {
    const int rc = map_check(B, S, H, KV, D);
    if (rc != HYC_OK) return rc;
    if (B == 0 || S == 0) return HYC_OK;
    if (!q || !k || !v || !o || !workspace) return HYC_ERR_NULL;
    if (!aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(o) || !aligned16(map) || !aligned16(workspace)) return HYC_ERR_ALIGN;
    if (mask && (!aligned16(mask) || mask_stride_b % 8 || mask_stride_row % 8)) return HYC_ERR_ALIGN;
    const MapWorkspace w = map_workspace(B, S, H);
    if (workspace_bytes < w.bytes) return HYC_ERR_WORKSPACE;
    MapArgs A = map_args(q, k, mask, mask_stride_b, mask_stride_row, threshold, workspace, B, S, H, KV, scale);
    A.v = (const uint16_t*)v; A.o = (uint16_t*)o; A.map = (uint16_t*)map;
    hipStream_t st = (hipStream_t)stream;
    if (mask) {
        const int mask_wgs = (int)cdiv(cdiv(S, 32) * cdiv(S, 512), 4), batches = mask_stride_b ? (int)B : 1;
        const dim3 wgs((unsigned)(mask_wgs * batches + cdiv(S, kMapTile) * B * KV));
        if (D == 128) map_classes_kernel<128><<<wgs, 256, 0, st>>>(A, mask_wgs, batches);
        else map_classes_kernel<64><<<wgs, 256, 0, st>>>(A, mask_wgs, batches);
    }
    const dim3 grid((unsigned)(cdiv(S, kMapRows) * B * H));
    if (D == 128) map_fwd_kernel<128><<<grid, 256, 0, st>>>(A);
    else map_fwd_kernel<64><<<grid, 256, 0, st>>>(A);
    if (threshold)
        map_row_scan_kernel<<<dim3((unsigned)cdiv(B * H * S, 1024)), 1024, 0, st>>>(A.counts, A.block_counts, B * H * S, (int)S,
                                                                                    const_cast<int64_t*>(A.row_offsets));
    return check_launch();
}

extern "C" int hyc_map_emit(const void* q, const void* k, const void* mask, int64_t mask_stride_b, int64_t mask_stride_row,
                            const float* threshold, const void* workspace, int64_t workspace_bytes, int64_t capacity, int64_t* indices,
                            void* values, int64_t* seg_offsets, int64_t B, int64_t S, int64_t H, int64_t KV, int64_t D, float scale,
                            void* stream) {
    const int rc = map_check(B, S, H, KV, D);
    if (rc != HYC_OK) return rc;
    if (capacity < 0) return HYC_ERR_SHAPE;
    if (B == 0 || S == 0) return HYC_OK;
    if (!q || !k || !threshold || !workspace || !seg_offsets || (capacity > 0 && (!indices || !values))) return HYC_ERR_NULL;
    if (!aligned16(q) || !aligned16(k) || !aligned16(workspace)) return HYC_ERR_ALIGN;
    if (mask && (!aligned16(mask) || mask_stride_b % 8 || mask_stride_row % 8)) return HYC_ERR_ALIGN;
    if (workspace_bytes < map_workspace(B, S, H).bytes) return HYC_ERR_WORKSPACE;
    MapArgs A = map_args(q, k, mask, mask_stride_b, mask_stride_row, threshold, const_cast<void*>(workspace), B, S, H, KV, scale);
    A.capacity = capacity; A.indices = indices; A.values = (uint16_t*)values; A.seg_offsets = seg_offsets;
    const dim3 grid((unsigned)(cdiv(S, kMapRows) * B * H));
    if (D == 128) map_emit_kernel<128><<<grid, 256, 0, (hipStream_t)stream>>>(A);
    else map_emit_kernel<64><<<grid, 256, 0, (hipStream_t)stream>>>(A);
    return check_launch();
}

extern "C" int64_t hyc_map_bwd_workspace(int64_t B, int64_t S, int64_t H, int64_t KV, int64_t D, int64_t capacity) {
    return B < 0 || S < 0 || H < 0 || D < 0 || capacity < 0 ? 0 : map_bwd_workspace(B, S, H, KV, D, capacity).bytes;
}

extern "C" int hyc_map_bwd(const void* grad_o, const void* q, const void* k, const void* v, const int64_t* indices, const void* values,
                           const int64_t* seg_offsets, int64_t capacity, void* workspace, int64_t workspace_bytes, void* grad_q,
                           void* grad_k, void* grad_v, int64_t B, int64_t S, int64_t H, int64_t KV, int64_t D, float scale, void* stream) {
    const int rc = map_check(B, S, H, KV, D);
    if (rc != HYC_OK) return rc;
    if (capacity < 0 || capacity >= (int64_t)1 << 31) return HYC_ERR_SHAPE;
    if (B == 0 || S == 0) return HYC_OK;
    if (!grad_o || !q || !k || !v || !seg_offsets || !workspace || !grad_q || !grad_k || !grad_v || (capacity > 0 && (!indices || !values)))
        return HYC_ERR_NULL;
    for (const void* p : {grad_o, q, k, v, (const void*)workspace, (const void*)grad_q, (const void*)grad_k, (const void*)grad_v})
        if (!aligned16(p)) return HYC_ERR_ALIGN;
    const MapBwdWorkspace w = map_bwd_workspace(B, S, H, KV, D, capacity);
    if (workspace_bytes < w.bytes) return HYC_ERR_WORKSPACE;
    char* ws = (char*)workspace;
    MapBwdArgs A = {};
    A.grad_o = (const uint16_t*)grad_o; A.q = (const uint16_t*)q; A.k = (const uint16_t*)k; A.v = (const uint16_t*)v;
    A.indices = indices; A.values = (const uint16_t*)values; A.seg_offsets = seg_offsets;
    A.entries = (uint32_t*)(ws + w.entries); A.grads = (uint16_t*)(ws + w.grads); A.tile_at = (uint32_t*)(ws + w.tile_at);
    A.wild = (uint32_t*)(ws + w.wild); A.wild_columns = (uint32_t*)(ws + w.wild_columns);
    A.grad_q = (uint16_t*)grad_q; A.grad_k = (uint16_t*)grad_k; A.grad_v = (uint16_t*)grad_v;
    if (H != KV) {
        A.grad_k = (uint16_t*)(ws + w.heads);
        A.grad_v = A.grad_k + (w.bytes - w.heads) / 4;
    }
    A.B = (int)B; A.S = (int)S; A.H = (int)H; A.KV = (int)KV; A.scale = scale;
    hipStream_t st = (hipStream_t)stream;
    const dim3 rows((unsigned)(cdiv(S, 32) * B * H)), blocks((unsigned)(cdiv(S, kMapRows) * B * H));
    map_regroup_kernel<<<rows, 256, 0, st>>>(A);
    if (D == 128) {
        map_bwd_q_kernel<128><<<blocks, 256, 0, st>>>(A);
        map_bwd_kv_kernel<128><<<blocks, 256, 0, st>>>(A);
    } else {
        map_bwd_q_kernel<64><<<blocks, 256, 0, st>>>(A);
        map_bwd_kv_kernel<64><<<blocks, 256, 0, st>>>(A);
    }
    if (H != KV) {
        const int64_t chunks = B * S * KV * D / 8;
        group_sum_kernel<<<dim3((unsigned)cdiv(chunks, 256), 2), 256, 0, st>>>(A.grad_k, A.grad_v, (uint16_t*)grad_k, (uint16_t*)grad_v, chunks,
                                                                              (int)(D / 8), (int)(H / KV));
    }
    return check_launch();
}
