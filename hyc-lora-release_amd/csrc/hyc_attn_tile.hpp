// Tiles of the attention kernels on the gfx950 matrix cores: staging of [rows, D] bf16 tiles in LDS with the
// asynchronous global -> LDS copies, and the two ways a v_mfma_f32_32x32x16_bf16 operand is read from such a tile.
//
// Operand layouts (lane l, half h = l / 32):
//   A [32 x 16]   lane l holds row l % 32, the eight k of its half h: k = 8h + j
//   B [16 x 32]   lane l holds column l % 32, k = 8h + j
//   C [32 x 32]   lane l holds column l % 32, register r: row 8*(r/4) + 4h + r%4
// A product whose C is the next product's B needs no exchange between lanes when the k of that next product are
// taken in the order the C registers hold them: registers 8t .. 8t+7 of a half are rows 16t + 4h + {0..3} and
// 16t + 8 + 4h + {0..3}.  The A operand of the next product must be read in the same order, which is what two
// transposing LDS reads (ds_read_b64_tr_b16: each 16 lanes fetch 4 rows x 16 columns and receive one column each)
// of rows 16t + 4h .. +3 and 16t + 8 + 4h .. +3 give.
#pragma once

#include "hyc_common.hpp"

namespace hyc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) char lds_char;

constexpr float kLog2e = 1.4426950408889634f;
constexpr float kLn2 = 0.6931471805599453f;

__device__ __forceinline__ bf16x8 as_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }
__device__ __forceinline__ f32x16 mfma32(bf16x8 a, bf16x8 b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ uint32_t lds_addr(const void* p) {
    return (uint32_t)(uintptr_t)(const lds_char*)p;
}

// 16 bytes per lane from base + voff (bytes) to LDS address lds + 16 * lane.  The copy is invisible to the compiler's
// counters: wait_copies() before the barrier that publishes the tile.
__device__ __forceinline__ void copy_to_lds16(const void* base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :: "s"(lds), "v"(voff), "s"(base) : "memory");
}
// 4 bytes per lane, to lds + 4 * lane
__device__ __forceinline__ void copy_to_lds4(const void* base, uint32_t voff, uint32_t lds) {
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                 :: "s"(lds), "v"(voff), "s"(base) : "memory");
}
__device__ __forceinline__ void wait_copies_and_barrier() {
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// A tile of ROWS rows of D bf16 in LDS.  The 16-byte chunks of a row are permuted so that neither read form meets bank
// conflicts: chunk c of row r lies at slot c ^ swz(r), which keeps pairs of chunks together (a transposing read takes
// 32 bytes of each of its 4 rows) and spreads 8 consecutive rows over different banks.  The copies write LDS in lane
// order, so the permutation is made by which chunk a lane fetches.
template <int D, int ROWS>
struct AttnTile {
    static constexpr int kChunks = D / 8;                       // 16-byte chunks of a row
    static constexpr int kPitch = D * 2;
    static constexpr int kBytes = ROWS * kPitch;
    static constexpr int kRowsPerCopy = 64 / kChunks;           // rows one wave instruction covers
    static constexpr int kCopies = ROWS / (kRowsPerCopy * 4);   // instructions of each of 4 waves

    __device__ static __forceinline__ int swz(int row) { return D == 128 ? 2 * (row & 7) : 2 * ((row >> 1) & 3); }

    // Requests rows row0 .. row0 + ROWS - 1 (past row_last: row_last again) of a tensor whose rows are `ld` elements
    // apart; called by the 4 waves of a workgroup.
    __device__ static __forceinline__ void request(const uint16_t* base, int row0, int row_last, int ld, uint32_t lds, int wave, int lane) {
        const int r_in = lane / kChunks, slot = lane % kChunks;
#pragma unroll
        for (int i = 0; i < kCopies; ++i) {
            const int row = (i * 4 + wave) * kRowsPerCopy + r_in;
            const int src = row0 + row < row_last ? row0 + row : row_last;
            const uint32_t voff = ((uint32_t)src * (uint32_t)ld + (uint32_t)((slot ^ swz(row)) * 8)) * 2u;
            copy_to_lds16(base, voff, lds + (uint32_t)((i * 4 + wave) * 1024));
        }
    }

    // A operand of rows r0 .. r0+31 (r0 a multiple of 32), k = columns 16t .. 16t+15
    __device__ static __forceinline__ bf16x8 rows_operand(const char* tile, int r0, int t, int lane) {
        const int row = lane & 31, h = lane >> 5;
        return as_bf16x8(*reinterpret_cast<const u32x4*>(tile + (r0 + row) * kPitch + (((2 * t + h) ^ swz(row)) * 16)));
    }
    // A operand of the transposed tile: rows = columns d0 .. d0+31 of the tile, k = tile rows k0 .. k0+15 (k0 a multiple
    // of 16) in the order 4h + {0..3}, 8 + 4h + {0..3}
    __device__ static __forceinline__ bf16x8 cols_operand(const char* tile, int k0, int d0, int lane) {
        const int i = lane & 15, g = (lane >> 4) & 1, h = lane >> 5;
        const int row = 4 * h + (i >> 2);                       // swz has period 8 in rows
        const int chunk = (d0 >> 3) + 2 * g + ((i & 3) >> 1);
        const char* p = tile + (k0 + row) * kPitch + (chunk ^ swz(row)) * 16 + (i & 1) * 8;
        typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(p + 8 * kPitch));
        const u32x2 a = __builtin_bit_cast(u32x2, lo), b = __builtin_bit_cast(u32x2, hi);
        return as_bf16x8(u32x4{a.x, a.y, b.x, b.y});
    }
};

// B operands of 32 rows of a row-major tensor (lane l: row l % 32), all D / 16 k steps
template <int D>
__device__ __forceinline__ void load_row_operands(const uint16_t* row, int h, bf16x8 (&v)[D / 16]) {
#pragma unroll
    for (int t = 0; t < D / 16; ++t) v[t] = as_bf16x8(ld16(row + 16 * t + 8 * h));
}

// Registers 8t .. 8t+7 of a C tile as the B operand of a following product (t = 0, 1)
__device__ __forceinline__ bf16x8 c_as_operand(const f32x16& c, int t) {
    u32x4 v;
#pragma unroll
    for (int p = 0; p < 4; ++p) v[p] = pk_bf16(c[8 * t + 2 * p], c[8 * t + 2 * p + 1]);
    return as_bf16x8(v);
}

// max / sum over the two halves of a wave, for every lane
__device__ __forceinline__ void half_values(float v, float& lo, float& hi) {
    const u32x2 r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, v), __builtin_bit_cast(uint32_t, v), false, false);
    const uint32_t a = r.x, b = r.y;                            // scalars first: a bit cast of a vector's element takes element 0
    lo = __builtin_bit_cast(float, a);
    hi = __builtin_bit_cast(float, b);
}
__device__ __forceinline__ float half_max(float v) {
    float a, b;
    half_values(v, a, b);
    return fmaxf(a, b);
}
__device__ __forceinline__ float half_sum(float v) {
    float a, b;
    half_values(v, a, b);
    return a + b;
}

// Stores a transposed C result (lane = row, registers = columns 32*db + 8*(r/4) + 4h + r%4) times `scale` as bf16
template <int D>
__device__ __forceinline__ void store_rows(uint16_t* row, int h, const f32x16 (&c)[D / 32], float scale) {
#pragma unroll
    for (int db = 0; db < D / 32; ++db)
#pragma unroll
        for (int b = 0; b < 4; ++b) {
            const u32x2 v = {pk_bf16(c[db][4 * b] * scale, c[db][4 * b + 1] * scale), pk_bf16(c[db][4 * b + 2] * scale, c[db][4 * b + 3] * scale)};
            st8(row + 32 * db + 8 * b + 4 * h, v);
        }
}

}  // namespace hyc
