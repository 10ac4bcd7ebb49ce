// The skinny LoRA products that stream a whole [T, N] tensor X for a rank-R result, for gfx950:
//
//   P1 = U^T . X   [R, N]   (contraction over the T rows;    U is [T, R])
//   P2 = X . V^T   [T, R]   (contraction over the N columns; V is [R, N])
//
// from ONE read of X, which is either dense bf16 or - for P1 - the packed codes of a compressed
// activation, dequantised in registers.  These are the four rank-R GEMMs of lora_forward /
// lora_backward (models/utils/compute_utils.py:22, :30-33):
//   x @ A                      P2 with V = A^T (the [R, in] layout nn.Linear keeps lora_A.weight in)
//   grad_y @ B^T, xa^T @ grad_y   P2 and P1 of the same X = grad_y in one pass
//   x^T @ grad_medium          P1, with x taken straight from its codes where the layer saved it
//                              compressed (the reference dequantises first,
//                              fused_llama_layer_intra_inter_full_fuse.py:375-383, :469-481).
// A library GEMM runs each of them at a fraction of the memory rate (output tiles 16 wide) and
// reads X once per product.  One launch takes the products of several projections: up to three X of
// one row count, or up to three rank-R products of one X (the codes of x are then read and decoded once).
//
// What bounds it: the read of X and, for small tensors, the two launches.  A wave has 16 KB of X on the
// way at any time and nothing else to wait for.
//
// Layout.  A workgroup of 4 waves owns a strip of rows and 512 columns; wave w keeps to the 128 columns
// 128w .. of them and walks down the strip, 16 rows a step, 4 steps of loads ahead.  So the sums of P1 stay
// in the wave's registers to the end of the strip, V is read once, and only P2 is added up across the
// four waves (through LDS, every 64 rows).  (Waves side by side along the rows, 64 rows each, had all their
// loads in one burst per tile and met at a barrier per tile for P1.)  X is held twice:
//   "chunk" form  lane (j = l%16, g = l/16): rows 4g .. 4g+3, columns 8j .. 8j+7  (16-byte loads)
//   "row"   form  lane (i = l%16, g = l/16): row i, columns 32s + 8g .. +7, s = 0..3
// P1 uses the chunk form as the B operand of v_mfma_f32_16x16x16_bf16 with permuted column slots
// (MFMA u takes column 8j + u of every lane), so a lane ends up with 8 consecutive columns of 4
// LoRA rows; P2 uses the row form as the A operand of v_mfma_f32_16x16x32_bf16, K running over the
// columns.  Only the chunk form is loaded from memory (256 contiguous bytes per row and instruction);
// the row form is the same tile turned through LDS, wave by wave.  U lies transposed in LDS, one 8-byte
// read an operand.
// Sums across strips (P1) and across column blocks (P2) go through fp32 partial planes that a small second
// kernel adds in order - no atomics, so results do not depend on scheduling - and rounds to bf16; where
// there is only one plane the results are written at once, and if that is so for all of them there is no
// second kernel (P1 of up to 256 rows).
#include <algorithm>
#include <type_traits>

#include "hyc_pack.hpp"

namespace hyc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kCtThreads = 256;
constexpr int kCtWaves = kCtThreads / kWave;
constexpr int kCtTile = 128;                              // columns per wave
constexpr int kCtBlock = kCtWaves * kCtTile;              // columns per workgroup
constexpr int kCtSub = 64;                                // rows between two sums of P2 across the waves; the shortest strip
constexpr int kCtSteps = kCtSub / 16;                     // steps of loads in flight
constexpr int kCtMaxStrip = 256;
constexpr int kCtPitch = kCtTile + 8;                     // LDS row pitch of a transposed tile (bf16 elements)
constexpr int kCtUPitch = kCtMaxStrip + 4;                // LDS pitch of a rank's column of U
constexpr int kCtMembers = 3;                             // X's in a launch, or rank-R products of one X
static Knob g_ct_strip{0};                                // rows of a strip, 0: by size; see hyc_set_tuning

struct ContractMember {
    const uint16_t* x;                   // dense X [T, N]
    const uint8_t* q;                    // or packed codes [T, N*q_bit/8] with
    const uint16_t* s; const uint16_t* zp;   //   steps / zero points bf16 [N]
    const uint16_t* u[4];                // per rank block of 16: [T, R], at the block's first rank
    const uint16_t* v[4];                // [R, N], or [N, R] with v_transposed, likewise
    uint16_t* p1[4]; uint16_t* p2[4];    // results, where there is one plane only
    float* part1;                        // [strips][16*blocks][N], or null
    float* part2;                        // [col_blocks][T][16*blocks], or null
    int N, C, v_transposed, p1_transposed, strip_rows;
    uint32_t col_blocks;
    uint32_t first_wg;
};
struct ContractArgs {
    ContractMember m[kCtMembers];
    int members, R, blocks;
    int live[4];                         // ranks of a block
    int64_t T;
};

__device__ __forceinline__ s16x4 pick_column(const u32x4 (&xv)[4], int u8) {
    // element u8 (0..7) of the four rows a lane holds in chunk form, as one MFMA operand
    const uint32_t sel = (u8 & 1) ? 0x07060302u : 0x05040100u;
    const int d = u8 >> 1;
    auto dw = [&](const u32x4& r) { return d == 0 ? r.x : (d == 1 ? r.y : (d == 2 ? r.z : r.w)); };
    const u32x2 pk = {__builtin_amdgcn_perm(dw(xv[1]), dw(xv[0]), sel), __builtin_amdgcn_perm(dw(xv[3]), dw(xv[2]), sel)};
    return __builtin_bit_cast(s16x4, pk);
}

// blockIdx.x: member, strip, column block; blockIdx.y: which NB rank blocks of 16 (ranks past 32 are covered by several
// workgroups, each reading X again, through the cache: every accumulator and operand scales with the blocks held at once)
template <int QBIT, bool ZP, bool P1, bool P2, int NB>
__global__ __launch_bounds__(kCtThreads) void lora_contract_kernel(const ContractArgs a) {
    static_assert(QBIT == 0 || !P2, "the column contraction reads dense X only");
    __shared__ __attribute__((aligned(16))) uint16_t ul[P1 ? NB * 16 * kCtUPitch : 8];
    __shared__ __attribute__((aligned(16))) uint16_t tr[P2 ? kCtWaves : 1][P2 ? 2 * 16 * kCtPitch : 8];
    __shared__ __attribute__((aligned(16))) float sum2[P1 ? 2 : 1][P2 ? kCtWaves * kCtSub * 16 * NB : 4];
    const int lane = threadIdx.x & (kWave - 1);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, g = lane >> 4;
    const uint32_t wg = blockIdx.x;
    const int mi = (a.members > 1 && wg >= a.m[1].first_wg ? 1 : 0) + (a.members > 2 && wg >= a.m[2].first_wg ? 1 : 0);
    const ContractMember& m = a.m[mi];
    const uint32_t local = wg - m.first_wg, in_strip = local / m.col_blocks;
    const int64_t strip = in_strip;
    const int cb = (int)(local - in_strip * m.col_blocks);
    const int b0 = blockIdx.y * NB;                             // first rank block
    const int N = m.N, R = a.R;
    const int64_t row0 = strip * m.strip_rows;
    const int rows = (int)(a.T - row0 < m.strip_rows ? a.T - row0 : m.strip_rows);
    const int c0 = cb * kCtBlock + wave * kCtTile;
    const int chunk = c0 / 8 + j;
    const bool active = chunk < m.C, full = c0 + kCtTile <= N;
    constexpr int QB = QBIT ? QBIT : 8;
    constexpr float kHalf = (float)(1 << (QB - 1));

    // Every load is issued whatever the lane (rows, columns and ranks past the end read the last one and are zeroed afterwards): a
    // load under a condition makes the compiler wait for all that is in flight at its next use.
    // U: thread (row t/8, rank pair t%8) of 32 rows an iteration; first in the queue, so that waiting for it leaves X in flight
    uint32_t uw[P1 ? NB : 1][P1 ? kCtMaxStrip / 32 : 1];
    const int up = threadIdx.x & 7, ur = threadIdx.x >> 3;
    if constexpr (P1) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int k = 0; k < kCtMaxStrip / 32; ++k) {
                const int r = 32 * k + ur < rows ? 32 * k + ur : rows - 1, rank = 2 * up < a.live[b0 + nb] ? 2 * up : 0;
                uw[nb][k] = *reinterpret_cast<const uint32_t*>(m.u[b0 + nb] + (row0 + r) * R + rank);
            }
    }
    // V operand of the column contraction: lane (rank j, g), columns c0 + 32s + 8g .. +7; [N, R]: the eight columns are R elements apart
    // (whole dwords, the wanted half picked afterwards: 16-bit loads into register halves would each wait for the one before)
    uint32_t e[P2 ? NB : 1][4][8];
    if constexpr (P2) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const int col = c0 + 32 * s + 8 * g < N ? c0 + 32 * s + 8 * g : 0;
                const int rank = j < a.live[b0 + nb] ? j : 0;
                if (m.v_transposed) {
                    const uint16_t* p = m.v[b0 + nb] + (int64_t)col * R + (rank & ~1);
#pragma unroll
                    for (int k = 0; k < 8; ++k) e[nb][s][k] = *reinterpret_cast<const uint32_t*>(p + k * R);
                } else {
                    const uint16_t* p = m.v[b0 + nb] + (int64_t)rank * N + col;
                    const u32x2 lo = ld8(p), hi = ld8(p + 4);
                    e[nb][s][0] = lo.x; e[nb][s][1] = lo.y; e[nb][s][2] = hi.x; e[nb][s][3] = hi.y;
                }
            }
    }
    // per-column constants of the dequantiser
    float sc[8], zz[8];
    const int ld_chunk = active ? chunk : m.C - 1;
    PackedSlot<QB> slot(ld_chunk);
    if constexpr (QBIT != 0) {
        unpack8(ld16(m.s + ld_chunk * 8), sc);
        if constexpr (ZP) unpack8(ld16(m.zp + ld_chunk * 8), zz);
    }
    // X of one step in chunk form
    u32x4 xv[kCtSteps][4];
    const int64_t x_pitch = QBIT == 0 ? 2 * (int64_t)N : (int64_t)N * QB / 8;
    const char* x_base = (QBIT == 0 ? (const char*)m.x + 16 * (int64_t)ld_chunk : (const char*)m.q + slot.offset) + row0 * x_pitch;
    auto load = [&](u32x4 (&dst)[4], int r0) {
#pragma unroll
        for (int vv = 0; vv < 4; ++vv) {
            const int r = r0 + 4 * g + vv < rows ? r0 + 4 * g + vv : rows - 1;
            const char* p = x_base + r * x_pitch;
            if constexpr (QBIT == 0) {
                dst[vv] = ld16(p);
            } else {
                const u32x2 w = ld8(p);
                dst[vv].x = w.x;
                dst[vv].y = w.y;
            }
        }
    };
#pragma unroll
    for (int st = 0; st < kCtSteps; ++st) load(xv[st], 16 * st);

    if constexpr (P1) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int k = 0; k < kCtMaxStrip / 32; ++k) {
                uint16_t* p = ul + (nb * 16 + 2 * up) * kCtUPitch + 32 * k + ur;
                const uint32_t w = 32 * k + ur < rows && 2 * up < a.live[b0 + nb] ? uw[nb][k] : 0u;
                p[0] = (uint16_t)w;
                p[kCtUPitch] = (uint16_t)(w >> 16);
            }
        __syncthreads();
    }
    u32x4 vop[P2 ? NB : 1][4];
    if constexpr (P2) {
        const uint32_t sel = (j & 1) ? 0x07060302u : 0x05040100u;         // high or low halves of two dwords
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                const auto& d = e[nb][s];
                vop[nb][s] = m.v_transposed ? u32x4{__builtin_amdgcn_perm(d[1], d[0], sel), __builtin_amdgcn_perm(d[3], d[2], sel),
                                                    __builtin_amdgcn_perm(d[5], d[4], sel), __builtin_amdgcn_perm(d[7], d[6], sel)}
                                            : u32x4{d[0], d[1], d[2], d[3]};
                if (!(j < a.live[b0 + nb] && c0 + 32 * s + 8 * g < N)) vop[nb][s] = u32x4{0, 0, 0, 0};
            }
    }

    f32x4 acc1[P1 ? NB : 1][8];
    if constexpr (P1) {
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int u8 = 0; u8 < 8; ++u8) acc1[nb][u8] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    }
    auto sub = [&](int base, int half, auto ahead_tag) __attribute__((always_inline)) {
        constexpr bool AHEAD = decltype(ahead_tag)::value;          // 64 more rows follow
        // two steps at a time, so that their chains through LDS and the matrix cores run side by side
#pragma unroll
        for (int s2 = 0; s2 < kCtSteps; s2 += 2) {
#pragma unroll
            for (int st = s2; st < s2 + 2; ++st) {
                const int r0 = base + 16 * st;
                if constexpr (QBIT != 0) {
#pragma unroll
                    for (int vv = 0; vv < 4; ++vv) {
                        float c[8], f[8];
                        slot.decode(u32x2{xv[st][vv].x, xv[st][vv].y}, c);
#pragma unroll
                        for (int e = 0; e < 8; ++e) {
                            if constexpr (ZP) f[e] = rbf((c[e] - kHalf) - zz[e]) * sc[e];
                            else f[e] = (c[e] - kHalf) * sc[e];
                        }
                        xv[st][vv] = pack8(f);
                    }
                }
                if (!full || r0 + 16 > rows) {                  // uniform: rows and columns past the end count as zeros
#pragma unroll
                    for (int vv = 0; vv < 4; ++vv)
                        if (!(active && r0 + 4 * g + vv < rows)) xv[st][vv] = u32x4{0, 0, 0, 0};
                }
                if constexpr (P2) {
                    // to the row form through this wave's corner of LDS: read straight from memory it would be 16 rows x 64
                    // bytes per load instruction
                    uint16_t* tw = tr[wave] + (st - s2) * 16 * kCtPitch;
#pragma unroll
                    for (int vv = 0; vv < 4; ++vv) *reinterpret_cast<u32x4*>(tw + (4 * g + vv) * kCtPitch + 8 * j) = xv[st][vv];
                }
            }
            if constexpr (P2) {
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
            }
            if constexpr (P1) {
#pragma unroll
                for (int st = s2; st < s2 + 2; ++st) {
                    s16x4 uop[NB];
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
                        uop[nb] = __builtin_bit_cast(s16x4, *reinterpret_cast<const u32x2*>(ul + (nb * 16 + j) * kCtUPitch + base + 16 * st + 4 * g));
#pragma unroll
                    for (int u8 = 0; u8 < 8; ++u8) {
                        const s16x4 xop = pick_column(xv[st], u8);
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb)
                            acc1[nb][u8] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(uop[nb], xop, acc1[nb][u8], 0, 0, 0);
                    }
                }
            }
            if constexpr (AHEAD) {
#pragma unroll
                for (int st = s2; st < s2 + 2; ++st) load(xv[st], base + 16 * st + kCtSub);
            }
            if constexpr (P2) {
                f32x4 acc2[2][NB];
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb) acc2[h][nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int s = 0; s < 4; ++s)
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        const bf16x8 xop = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4*>(tr[wave] + (16 * h + j) * kCtPitch + 32 * s + 8 * g));
#pragma unroll
                        for (int nb = 0; nb < NB; ++nb)
                            acc2[h][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xop, __builtin_bit_cast(bf16x8, vop[nb][s]), acc2[h][nb], 0, 0, 0);
                    }
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                        for (int vv = 0; vv < 4; ++vv)
                            sum2[half][((wave * kCtSub + 16 * (s2 + h) + 4 * g + vv) * NB + nb) * 16 + j] = acc2[h][nb][vv];
            }
        }
        if constexpr (P2) {
            // the waves' parts of 64 rows, added in wave order (zeros from a wave past the last column): thread t owns 4 ranks of
            // NB (row, block) pairs
            __syncthreads();
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const int i = k * kCtThreads + threadIdx.x;
                const int row = i / (4 * NB), nb = (i >> 2) % NB, r4 = (i & 3) * 4;
                f32x4 s = *reinterpret_cast<const f32x4*>(sum2[half] + (row * NB + nb) * 16 + r4);
#pragma unroll
                for (int w = 1; w < kCtWaves; ++w) s += *reinterpret_cast<const f32x4*>(sum2[half] + ((w * kCtSub + row) * NB + nb) * 16 + r4);
                if (base + row < rows) {
                    const int64_t t = row0 + base + row;
                    if (m.part2) {
                        *reinterpret_cast<f32x4*>(m.part2 + ((int64_t)cb * a.T + t) * (16 * a.blocks) + 16 * (b0 + nb) + r4) = s;
                    } else {
                        uint32_t* p = reinterpret_cast<uint32_t*>(m.p2[b0 + nb] + t * R + r4);
                        if (r4 < a.live[b0 + nb]) p[0] = pk_bf16(s.x, s.y);
                        if (r4 + 2 < a.live[b0 + nb]) p[1] = pk_bf16(s.z, s.w);
                    }
                }
            }
        }
    };
    int base = 0, half = 0;                                     // half of sum2: with two, one barrier per 64 rows is enough
    if constexpr (P1)                                           // without P1 a strip is 64 rows
        for (; base + kCtSub < rows; base += kCtSub, half ^= 1) sub(base, half, std::true_type{});
    sub(base, half, std::false_type{});

    if constexpr (P1) {
        if (!active) return;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            if (m.part1) {
#pragma unroll
                for (int vv = 0; vv < 4; ++vv) {
                    float* dst = m.part1 + (strip * (16 * a.blocks) + 16 * (b0 + nb) + 4 * g + vv) * (int64_t)N + chunk * 8;
                    float e[8];
#pragma unroll
                    for (int u8 = 0; u8 < 8; ++u8) e[u8] = acc1[nb][u8][vv];
                    *reinterpret_cast<f32x4*>(dst) = f32x4{e[0], e[1], e[2], e[3]};
                    *reinterpret_cast<f32x4*>(dst + 4) = f32x4{e[4], e[5], e[6], e[7]};
                }
            } else if (m.p1_transposed) {
#pragma unroll
                for (int u8 = 0; u8 < 8; ++u8) {
                    uint32_t* p = reinterpret_cast<uint32_t*>(m.p1[b0 + nb] + (int64_t)(chunk * 8 + u8) * R + 4 * g);
                    const f32x4 s = acc1[nb][u8];
                    if (4 * g < a.live[b0 + nb]) p[0] = pk_bf16(s.x, s.y);
                    if (4 * g + 2 < a.live[b0 + nb]) p[1] = pk_bf16(s.z, s.w);
                }
            } else {
#pragma unroll
                for (int vv = 0; vv < 4; ++vv) {
                    float e[8];
#pragma unroll
                    for (int u8 = 0; u8 < 8; ++u8) e[u8] = acc1[nb][u8][vv];
                    uint32_t* p = reinterpret_cast<uint32_t*>(m.p1[b0 + nb] + (int64_t)(4 * g + vv) * N + chunk * 8);
                    if (4 * g + vv < a.live[b0 + nb]) {
#pragma unroll
                        for (int h = 0; h < 4; ++h) p[h] = pk_bf16(e[2 * h], e[2 * h + 1]);
                    }
                }
            }
        }
    }
}

// P2 alone, for X of many rows or few columns: a workgroup of 8 waves owns 16 rows and the whole contraction, so there are no
// partial planes and no second kernel.  A wave takes 128 of every 1024 columns, 32 (64 bytes of a row) an operand.  X and V are
// read four neighbouring lanes to a row's 64 bytes, and the operands (lane (i, g): row i, columns 8g .. +7 of the 32) come of that by a
// lane permutation: in the operands' own order neighbouring lanes are in 16 rows, and the cache takes a cycle for each.  Two
// turns of loads are on their way.
constexpr int kRowsThreads = 512, kRowsWaves = kRowsThreads / kWave, kRowsCols = kRowsWaves * kCtTile;
template <int NB>
__global__ __launch_bounds__(kRowsThreads, 2) void lora_rows_kernel(const ContractArgs a) {
    constexpr int kAhead = 2;
    __shared__ float part[kRowsWaves][NB * 256];
    const ContractMember& m = a.m[0];
    const int lane = threadIdx.x & (kWave - 1), wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4, N = m.N, R = a.R, b0 = blockIdx.y * NB;
    const int64_t row0 = (int64_t)blockIdx.x * 16;
    const int rows = a.T - row0 < 16 ? (int)(a.T - row0) : 16;
    const int lr = lane >> 2, lc = 8 * (lane & 3);
    const uint16_t* xp = m.x + (row0 + (lr < rows ? lr : rows - 1)) * N + lc;       // rows past the end: not stored
    const uint16_t* vp[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) vp[nb] = m.v[b0 + nb] + (int64_t)(lr < a.live[b0 + nb] ? lr : 0) * N + lc;
    u32x4 x[kAhead][4], v[kAhead][NB][4];
    auto load = [&](int d, int c0) __attribute__((always_inline)) {
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            const int c = c0 + 32 * s < N ? c0 + 32 * s : 0;                        // uniform; columns past the end: not multiplied
            x[d][s] = ld16(xp + c);
#pragma unroll
            for (int nb = 0; nb < NB; ++nb) v[d][nb][s] = ld16(vp[nb] + c);
        }
    };
    auto operand = [&](u32x4 w) __attribute__((always_inline)) {
#pragma unroll
        for (int d = 0; d < 4; ++d) w[d] = (uint32_t)__builtin_amdgcn_ds_bpermute(4 * (4 * i + g), (int)w[d]);
        return __builtin_bit_cast(bf16x8, w);
    };
    f32x4 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    const int w0 = wave * kCtTile;
#pragma unroll
    for (int d = 0; d < kAhead; ++d) load(d, w0 + d * kRowsCols);
    for (int c0 = w0; c0 < N; c0 += kAhead * kRowsCols) {
#pragma unroll
        for (int d = 0; d < kAhead; ++d) {
            const int c = c0 + d * kRowsCols;
            bf16x8 xo[4], vo[NB][4];
#pragma unroll
            for (int s = 0; s < 4; ++s) {
                xo[s] = operand(c + 32 * s < N ? x[d][s] : u32x4{0, 0, 0, 0});
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) vo[nb][s] = operand(c + 32 * s < N ? v[d][nb][s] : u32x4{0, 0, 0, 0});
            }
            load(d, c + kAhead * kRowsCols);
#pragma unroll
            for (int s = 0; s < 4; ++s)
#pragma unroll
                for (int nb = 0; nb < NB; ++nb) acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(xo[s], vo[nb][s], acc[nb], 0, 0, 0);
        }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int e = 0; e < 4; ++e) part[wave][nb * 256 + (4 * g + e) * 16 + i] = acc[nb][e];
    __syncthreads();
    // the waves' parts in wave order; a thread owns two ranks of a row
    for (int o = threadIdx.x; o < NB * 128; o += kRowsThreads) {
        const int nb = o >> 7, row = (o >> 3) & 15, r = (o & 7) * 2;
        float s0 = part[0][nb * 256 + row * 16 + r], s1 = part[0][nb * 256 + row * 16 + r + 1];
#pragma unroll
        for (int w = 1; w < kRowsWaves; ++w) {
            s0 += part[w][nb * 256 + row * 16 + r];
            s1 += part[w][nb * 256 + row * 16 + r + 1];
        }
        if (row < rows && r < a.live[b0 + nb]) *reinterpret_cast<uint32_t*>(m.p2[b0 + nb] + (row0 + row) * R + r) = pk_bf16(s0, s1);
    }
}

// out[i][c] = bf16( sum_k part[k][i][c] ), i < rows_out, c < cols_out, partial planes of
// [rows_part][cols_part] floats; up to six such reductions per launch.  Bound by latency: a block takes 64 vectors of W
// floats and each of its waves a quarter of the planes, up to 8 loads in flight, and the quarters meet in LDS in
// plane order (one thread for all planes of a vector: 6 us for 32 planes of [16, 4096], of which 4 waiting).
struct ReduceJob {
    const float* part; uint16_t* out;
    int64_t rows_out, plane;                  // plane: floats from one plane to the next
    int cols_out, cols_part, planes;
    int transposed;          // out is [cols_out][rows_out]: rows_out <= 64 and even, cols_out % 4 == 0
    int64_t first_block;
};
constexpr int kReduceJobs = 2 * kCtMembers;
struct ReduceArgs { ReduceJob j[kReduceJobs]; int jobs; };
constexpr int kReduceWaves = 4;
template <int W>
__global__ __launch_bounds__(256) void contract_reduce_kernel(const ReduceArgs a) {
    typedef float fvec __attribute__((ext_vector_type(W)));
    __shared__ __attribute__((aligned(16))) float quarter[kReduceWaves][kWave * W];
    int ji = 0;
    for (int k = 1; k < a.jobs; ++k) ji += (int64_t)blockIdx.x >= a.j[k].first_block ? 1 : 0;
    const ReduceJob& jb = a.j[ji];
    const int64_t blk = blockIdx.x - jb.first_block;
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    // a block's vectors: 64 in a row, or (transposed) W columns x 16 lanes of 4 rows
    const uint32_t col_groups = (uint32_t)(jb.cols_out + 16 * W - 1) / (16 * W);
    const uint32_t tr4 = (uint32_t)blk / col_groups;
    const int64_t tr0 = (int64_t)tr4 * 4, tc0 = (int64_t)((uint32_t)blk - tr4 * col_groups) * (16 * W);
    const int64_t idx = (blk * kWave + lane) * W;             // cols_out % W == 0: a vector lies in one row
    // (a 64-bit division takes longer than the loads)
    const bool small = jb.rows_out * jb.cols_out <= UINT32_MAX;
    const int64_t row = jb.transposed ? tr0 + (lane >> 4) : small ? (int64_t)((uint32_t)idx / (uint32_t)jb.cols_out) : idx / jb.cols_out;
    const int64_t col = jb.transposed ? tc0 + (lane & 15) * W : idx - row * jb.cols_out;
    const bool valid = row < jb.rows_out && col < jb.cols_out;
    // a wave's share is a run of planes, eight of them in flight
    const float* p = jb.part + row * jb.cols_part + col;
    const int share = (jb.planes + kReduceWaves - 1) / kReduceWaves;
    const int k0 = wave * share, k1 = k0 + share < jb.planes ? k0 + share : jb.planes;
    float sum[W];
#pragma unroll
    for (int e = 0; e < W; ++e) sum[e] = 0.0f;
    if (valid)
        for (int k = k0; k < k1; k += 8) {
            fvec v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = *reinterpret_cast<const fvec*>(p + (k + u < k1 ? k + u : k1 - 1) * jb.plane);
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int e = 0; e < W; ++e) sum[e] += k + u < k1 ? v[u][e] : 0.0f;
        }
#pragma unroll
    for (int e = 0; e < W; ++e) quarter[wave][lane * W + e] = sum[e];
    __syncthreads();
    if (wave != 0) return;
    if (jb.transposed) {
        // lane = a column, whose 4 ranks leave together
        for (int c = lane; c < 16 * W; c += kWave) {
            if (tc0 + c >= jb.cols_out) continue;
            float t[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                t[r] = quarter[0][r * 16 * W + c];
#pragma unroll
                for (int w = 1; w < kReduceWaves; ++w) t[r] += quarter[w][r * 16 * W + c];
            }
            uint32_t* out = reinterpret_cast<uint32_t*>(jb.out + (tc0 + c) * jb.rows_out + tr0);
            out[0] = pk_bf16(t[0], t[1]);
            if (tr0 + 2 < jb.rows_out) out[1] = pk_bf16(t[2], t[3]);
        }
        return;
    }
    if (!valid) return;
#pragma unroll
    for (int w = 1; w < kReduceWaves; ++w)
#pragma unroll
        for (int e = 0; e < W; ++e) sum[e] += quarter[w][lane * W + e];
    uint32_t* out = reinterpret_cast<uint32_t*>(jb.out + idx);
#pragma unroll
    for (int e = 0; e < W; e += 2) out[e / 2] = pk_bf16(sum[e], sum[e + 1]);
}

// ------------------------------------------------------------------------------------
template <int QBIT, bool ZP, bool P1, bool P2>
static void contract_launch(const ContractArgs& a, int64_t wgs, hipStream_t st) {
    // rank blocks held at once: all of up to three, two of four; both products of three take one at a time
    const dim3 block(kCtThreads);
    const int nb = a.blocks == 4 ? 2 : (P1 && P2 && a.blocks == 3 ? 1 : a.blocks);
    const dim3 grid((unsigned)wgs, (unsigned)(a.blocks / nb));
    if (nb == 1) hipLaunchKernelGGL((lora_contract_kernel<QBIT, ZP, P1, P2, 1>), grid, block, 0, st, a);
    else if (nb == 2) hipLaunchKernelGGL((lora_contract_kernel<QBIT, ZP, P1, P2, 2>), grid, block, 0, st, a);
    else if constexpr (!(P1 && P2)) hipLaunchKernelGGL((lora_contract_kernel<QBIT, ZP, P1, P2, 3>), grid, block, 0, st, a);
}

// Rows of a strip: 256 where that leaves 160 workgroups and more or is all there is, 64 where even those are 64 workgroups and less, else 128.
// Fewer strips are fewer planes of P1 (2 x 16 N x 4 bytes each), more strips more units at work: both products at 128 and 256 rows [T, N],
// us: [4096, 11008] 32.1 / 30.2 (352 workgroups at 256), [2040, 13824] 22.5 / 20.3 (216), [2048, 11008] 21.0 / 18.2 (176), [4096, 4096] 16.6 / 17.2
// (128), [2040, 5120] 15.5 / 16.3 (80), [2048, 4096] 14.9 / 16.0 (64);  at 64 and 128 rows, both products and P1 from codes: [300, 768] 8.5 / 9.9 and 8.4 /
// 9.6 (10 workgroups at 64), [1000, 2048] 9.4 / 10.4 and 9.2 / 10.2 (64), [4096, 96] 9.1 / 10.1 and 9.2 / 10.8 (64), [680, 4096] 10.0 / 10.7 and 10.1 / 10.3 (88),
// but three projections in a launch 32 / 29 there, 24 / 25 at [300, 4096] (40), 20.8 / 23.2 at [1000, 768] (32).  It depends on T and N alone, so
// that the sums are in one order whatever else is in the launch and whatever X is read from.
// Without P1 a strip leaves nothing behind, and 64 rows are the fastest at every shape measured ([4096, 11008] 24.5 against 26.5 at 256,
// [512, 4096] 7.6 against 11.4).
static int strip_rows(int64_t T, int64_t N, bool want1) {
    if (!want1) return kCtSub;
    const int fixed = g_ct_strip.get();
    if (fixed) return fixed;
    const int64_t col_blocks = cdiv(N, kCtBlock);
    if (T <= kCtMaxStrip || cdiv(T, kCtMaxStrip) * col_blocks >= 160) return kCtMaxStrip;
    return cdiv(T, kCtSub) * col_blocks <= 64 ? kCtSub : 128;
}

// Whether x V^T alone goes to the kernel that keeps whole rows to a workgroup: up to 4096 columns, V as it lies.  That kernel against
// the planes and their sum, us (16 ranks): [4096, 768] 4.2 / 7.8, [96, 4096] 4.8 / 6.2, [512, 4096] 6.0 / 7.7, [4096, 4096] 10.4 / 13.2, [8192, 4096]
// 17.4 / 19.5;  from 5120 columns on the rows' serial chain is the longer: [2048, 5120] 12.5 / 11.6, [96, 11008] 12.4 / 7.6, [2048, 11008]
// 21.3 / 14.7, [4096, 11008] 25.4 / 23.2.
static bool whole_rows(const hyc_contract_job* jobs, int count, int64_t T) {
    for (int i = 0; i < count; ++i)
        if (jobs[i].v_transposed || !aligned16(jobs[i].v)) return false;
    return jobs[0].N <= 4096 && cdiv(T, 16) <= INT32_MAX;
}

int tune_contract(const char* key, int value) {
    if (strcmp(key, "contract_max_groups") == 0)              // without effect; accepted from callers that set it
        return value < 1 || value > 65536 ? HYC_ERR_ARG : HYC_OK;
    if (strcmp(key, "contract_strip_rows") == 0) {
        if (value < 0 || value > kCtMaxStrip || value % kCtSub) return HYC_ERR_ARG;
        g_ct_strip.set(value);
        return HYC_OK;
    }
    return 1;
}

// `count` products of X's of their own, or (`shared`) of the X of the first; one rank R for all, up to 16 where there are several
static int contract_jobs(const hyc_contract_job* jobs, int count, bool shared, int q_bit, void* workspace, int64_t workspace_bytes,
                         int64_t T, int64_t R, hipStream_t st) {
    const hyc_contract_job& h = jobs[0];
    const bool codes = h.q != nullptr, want1 = h.p1 != nullptr, want2 = h.p2 != nullptr;
    if (codes && q_bit != 2 && q_bit != 4 && q_bit != 8) return HYC_ERR_QBIT;
    if (T < 0 || T > ((int64_t)1 << 40)) return HYC_ERR_SHAPE;
    if (R < 2 || R > 64 || R % 2 != 0 || (count > 1 && R > 16)) return HYC_ERR_RANK;
    if (!want1 && !want2) return HYC_ERR_NULL;
    for (int i = 0; i < count; ++i) {
        const hyc_contract_job& jb = jobs[i];
        if (jb.N < 0 || jb.N % 32 != 0 || jb.N > (1 << 28)) return HYC_ERR_SHAPE;
        if ((jb.p1 != nullptr) != want1 || (jb.p2 != nullptr) != want2 || (want1 && !jb.u) || (want2 && !jb.v)) return HYC_ERR_NULL;
        if (i && shared && (jb.N != h.N || jb.v_transposed != h.v_transposed || jb.p1_transposed != h.p1_transposed)) return HYC_ERR_ARG;
        if (i == 0 || !shared) {
            if (codes ? (jb.x != nullptr || !jb.q || !jb.scale || want2 || (jb.zero_point != nullptr) != (h.zero_point != nullptr))
                      : (jb.x == nullptr || jb.q != nullptr))
                return HYC_ERR_ARG;
        }
    }
    if (!workspace) return HYC_ERR_NULL;
    for (int i = 0; i < count; ++i)
        if (T * jobs[i].N == 0) {
            if (count == 1) return HYC_OK;
            return HYC_ERR_SHAPE;
        }
    auto off = [](const void* p, uintptr_t by) { return p && (reinterpret_cast<uintptr_t>(p) & (by - 1)) != 0; };
    for (int i = 0; i < count; ++i) {
        const hyc_contract_job& jb = jobs[i];
        if (off(jb.x, 16) || off(jb.scale, 16) || off(jb.zero_point, 16) || off(jb.q, 8) || off(jb.v, 8) || off(jb.u, 4) || off(jb.p1, 4) ||
            off(jb.p2, 4))
            return HYC_ERR_ALIGN;
    }
    if (!aligned16(workspace)) return HYC_ERR_ALIGN;

    ContractArgs a{};
    ReduceArgs ra{};
    a.T = T; a.R = (int)R; a.members = shared ? 1 : count;
    a.blocks = shared ? count : (int)cdiv(R, 16);
    for (int b = 0; b < 4; ++b) a.live[b] = shared ? (int)R : (int)std::min<int64_t>(16, std::max<int64_t>(0, R - 16 * b));
    if (want2 && !want1 && a.members == 1 && whole_rows(jobs, shared ? count : 1, T)) {
        ContractMember& m = a.m[0];
        m.x = (const uint16_t*)h.x; m.N = (int)h.N;
        for (int b = 0; b < a.blocks; ++b) {
            m.v[b] = (const uint16_t*)(shared ? jobs[b].v : h.v) + (shared ? 0 : 16 * b * h.N);
            m.p2[b] = (uint16_t*)(shared ? jobs[b].p2 : h.p2) + (shared ? 0 : 16 * b);
        }
        const int nb = a.blocks == 4 ? 2 : a.blocks;
        const dim3 grid((unsigned)cdiv(T, 16), (unsigned)(a.blocks / nb)), block(kRowsThreads);
        if (nb == 1) hipLaunchKernelGGL(lora_rows_kernel<1>, grid, block, 0, st, a);
        else if (nb == 2) hipLaunchKernelGGL(lora_rows_kernel<2>, grid, block, 0, st, a);
        else hipLaunchKernelGGL(lora_rows_kernel<3>, grid, block, 0, st, a);
        return check_launch();
    }
    const int64_t rows16 = 16 * a.blocks;
    char* ws = (char*)workspace;
    int64_t used = 0, wgs = 0, rblocks = 0;
    const int w = (want2 && R % 4 != 0) ? 2 : 4;             // N % 32 == 0; R is even
    auto reduce = [&](const float* part, uint16_t* out, int64_t rows_out, int64_t plane, int64_t cols_out, int64_t cols_part, int64_t planes, int transposed) {
        ReduceJob& jb = ra.j[ra.jobs++];
        jb.part = part; jb.out = out; jb.rows_out = rows_out; jb.plane = plane; jb.cols_out = (int)cols_out; jb.cols_part = (int)cols_part;
        jb.planes = (int)planes; jb.transposed = transposed; jb.first_block = rblocks;
        rblocks += transposed ? cdiv(rows_out, 4) * cdiv(cols_out, 16 * w) : cdiv(rows_out * cols_out, kWave * w);
    };
    for (int i = 0; i < a.members; ++i) {
        const hyc_contract_job& jb = jobs[i];
        ContractMember& m = a.m[i];
        m.x = (const uint16_t*)jb.x; m.q = (const uint8_t*)jb.q; m.s = (const uint16_t*)jb.scale; m.zp = (const uint16_t*)jb.zero_point;
        m.N = (int)jb.N; m.C = (int)(jb.N / 8); m.v_transposed = jb.v_transposed; m.p1_transposed = jb.p1_transposed;
        m.col_blocks = (int)cdiv(jb.N, kCtBlock);
        m.strip_rows = strip_rows(T, jb.N, want1);
        const int64_t strips = cdiv(T, m.strip_rows);
        m.first_wg = (uint32_t)wgs;
        wgs += strips * m.col_blocks;
        if (want1 && strips > 1) { m.part1 = (float*)(ws + used); used += strips * rows16 * jb.N * 4; }
        if (want2 && m.col_blocks > 1) { m.part2 = (float*)(ws + used); used += (int64_t)m.col_blocks * T * rows16 * 4; }
        for (int b = 0; b < a.blocks; ++b) {
            const hyc_contract_job& from = shared ? jobs[b] : jb;
            const int64_t r = shared ? 0 : 16 * b;           // first rank of the block in its operands
            if (from.u) m.u[b] = (const uint16_t*)from.u + r;
            if (from.v) m.v[b] = (const uint16_t*)from.v + (from.v_transposed ? r : r * jb.N);
            if (from.p1) m.p1[b] = (uint16_t*)from.p1 + (from.p1_transposed ? r : r * jb.N);
            if (from.p2) m.p2[b] = (uint16_t*)from.p2 + r;
        }
        for (int b = 0; b < (shared ? count : 1); ++b) {     // the ranks of one result lie together, whatever blocks they were formed in
            if (m.part1) reduce(m.part1 + 16 * b * jb.N, (uint16_t*)jobs[shared ? b : i].p1, R, rows16 * jb.N, jb.N, jb.N, strips, jb.p1_transposed);
            if (m.part2) reduce(m.part2 + 16 * b, (uint16_t*)jobs[shared ? b : i].p2, T, T * rows16, R, rows16, m.col_blocks, 0);
        }
    }
    if (workspace_bytes < used) return HYC_ERR_ARG;
    if (wgs > INT32_MAX || rblocks > INT32_MAX) return HYC_ERR_SHAPE;
    if (codes) {
        const bool zp = h.zero_point != nullptr;
#define HYC_CT_CODES(QB)                                                        \
        do {                                                                    \
            if (zp) contract_launch<QB, true, true, false>(a, wgs, st);         \
            else contract_launch<QB, false, true, false>(a, wgs, st);           \
        } while (0)
        if (q_bit == 8) HYC_CT_CODES(8);
        else if (q_bit == 4) HYC_CT_CODES(4);
        else HYC_CT_CODES(2);
#undef HYC_CT_CODES
    } else if (want1 && want2) {
        contract_launch<0, false, true, true>(a, wgs, st);
    } else if (want1) {
        contract_launch<0, false, true, false>(a, wgs, st);
    } else {
        contract_launch<0, false, false, true>(a, wgs, st);
    }
    if (ra.jobs == 0) return check_launch();
    if (hipGetLastError() != hipSuccess) return HYC_ERR_LAUNCH;
    if (w == 4) hipLaunchKernelGGL(contract_reduce_kernel<4>, dim3((unsigned)rblocks), dim3(256), 0, st, ra);
    else hipLaunchKernelGGL(contract_reduce_kernel<2>, dim3((unsigned)rblocks), dim3(256), 0, st, ra);
    return check_launch();
}

}  // namespace hyc

using namespace hyc;

extern "C" int64_t hyc_lora_contract_workspace(int64_t T, int64_t N, int64_t R, int want_p1, int want_p2) {
    if (T <= 0 || N <= 0 || R < 2 || R > 64) return 0;
    const int64_t strips = cdiv(T, strip_rows(T, N, want_p1 != 0)), cols = cdiv(N, kCtBlock), rows16 = 16 * cdiv(R, 16);
    int64_t bytes = 0;
    if (want_p1 && strips > 1) bytes += strips * rows16 * N * 4;
    if (want_p2 && cols > 1) bytes += cols * T * rows16 * 4;
    return bytes;
}

extern "C" int hyc_lora_contract(const void* x, const void* q, const void* scale, const void* zero_point, int q_bit,
                                 const void* u, const void* v, int v_transposed, void* p1, int p1_transposed, void* p2,
                                 void* workspace, int64_t workspace_bytes, int64_t T, int64_t N, int64_t R,
                                 void* stream) {
    const hyc_contract_job job = {x, q, scale, zero_point, u, v, p1, p2, N, v_transposed, p1_transposed};
    return contract_jobs(&job, 1, false, q_bit, workspace, workspace_bytes, T, R, (hipStream_t)stream);
}

extern "C" int hyc_lora_contract_group(const hyc_contract_job* jobs, int count, int shared, int q_bit, void* workspace,
                                       int64_t workspace_bytes, int64_t T, int64_t R, void* stream) {
    if (!jobs) return HYC_ERR_NULL;
    if (count < 1 || count > kCtMembers) return HYC_ERR_ARG;
    return contract_jobs(jobs, count, shared != 0 && count > 1, q_bit, workspace, workspace_bytes, T, R, (hipStream_t)stream);
}
