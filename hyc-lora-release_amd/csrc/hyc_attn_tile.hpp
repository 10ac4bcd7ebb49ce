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

// The same while the N youngest copies of the wave stay under way
template <int N>
__device__ __forceinline__ void wait_older_copies_and_barrier() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}

// A tile of ROWS rows of D bf16 in LDS, as 1 KB blocks of 16 rows x 4 chunks (of 16 bytes): block (row / 16, chunk / 4),
// inside it the 64 bytes of a row together, its chunks in the order chunk ^ (row / 4).  A wave's copy fills one block, four
// neighbouring lanes 64 contiguous bytes of memory: with the lanes of a row 16 apart (chunk-major blocks) the copies found 64
// lines instead of 16 per instruction and moved 28 bytes per ns and unit, a quarter of what L2 gives.  An operand of 32
// rows reads a chunk of 16 rows, a transposing read 4 rows of 4 chunks; both meet 256 bytes of different banks.  Everything
// that varies inside a kernel's loops (k step, column block, buffer) moves the address by a multiple of a block, an immediate
// offset: four registers of addresses serve all reads.
template <int D, int ROWS>
struct AttnTile {
    static constexpr int kChunks = D / 8;                       // 16-byte chunks of a row
    static constexpr int kBlocksAcross = kChunks / 4;
    static constexpr int kBytes = ROWS * D * 2;
    static constexpr int kCopies = kBytes / 4096;               // block copies of each of 4 waves

    // Bytes of chunk c (0..3) of row r (0..15) in a block
    __device__ static __forceinline__ int in_block(int r, int c) { return r * 64 + ((c ^ (r >> 2)) * 16); }

    // Requests rows row0 .. row0 + ROWS - 1 (past row_last: row_last again) of a tensor whose rows are `ld` elements
    // apart; called by the 4 waves of a workgroup.
    __device__ static __forceinline__ void request(const uint16_t* base, int row0, int row_last, int ld, uint32_t lds, int wave, int lane) {
#pragma unroll
        for (int i = 0; i < kCopies; ++i) {
            const int blk = i * 4 + wave;
            copy_to_lds16(base, source(blk, row0, row_last, ld, lane), lds + (uint32_t)(blk * 1024));
        }
    }
    // Bytes from the tensor's base to what a lane copies into block `blk`
    __device__ static __forceinline__ uint32_t source(int blk, int row0, int row_last, int ld, int lane) {
        const int r = lane >> 2, c = (lane & 3) ^ (r >> 2), row = (blk / kBlocksAcross) * 16 + r;
        const int src = row0 + row < row_last ? row0 + row : row_last;
        return ((uint32_t)src * (uint32_t)ld + (uint32_t)((blk % kBlocksAcross) * 32 + c * 8)) * 2u;
    }

    // What a lane adds to a tile's LDS address for the two read forms
    struct Lane {
        uint32_t rows[2], cols[2], order[4];
        __device__ __forceinline__ explicit Lane(int lane) {
            const int h = lane >> 5, r16 = lane & 15, rb = (lane >> 4) & 1;
#pragma unroll
            for (int odd = 0; odd < 2; ++odd) {
                const int c = 2 * odd + h;
                rows[odd] = (uint32_t)(rb * kBlocksAcross * 1024 + in_block(r16, c));
                const int row = 4 * h + (r16 >> 2) + 8 * odd, cc = 2 * rb + ((r16 & 3) >> 1);
                cols[odd] = (uint32_t)(in_block(row, cc) + (r16 & 1) * 8);
            }
#pragma unroll
            for (int c = 0; c < 4; ++c) order[c] = (uint32_t)(rb * kBlocksAcross * 1024 + in_block(r16, c) + h * 8);
        }
    };
    // The lane's addresses in one tile, opaque so that what a read adds to them stays an immediate offset instead of an
    // addition each (a third of the forward kernel's integer instructions)
    __device__ static __forceinline__ Lane in_tile(const Lane& at, uint32_t tile) {
        Lane v(at);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            v.rows[i] += tile; v.cols[i] += tile;
            asm("" : "+v"(v.rows[i]), "+v"(v.cols[i]));
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) v.order[i] += tile;
        return v;
    }
    // A operand of tile rows r0 .. r0+31 (r0 a multiple of 32), k = columns 16t .. 16t+15; `off`: constant bytes past the tile
    __device__ static __forceinline__ bf16x8 rows_operand(const Lane& at, int off, int r0, int t) {
        typedef const __attribute__((address_space(3))) u32x4 lds_u32x4;
        return as_bf16x8(*(lds_u32x4*)(at.rows[t & 1] + (uint32_t)(off + ((r0 / 16) * kBlocksAcross + t / 2) * 1024)));
    }
    // The same rows and k in the order 4h + {0..3}, 8 + 4h + {0..3}: the other operand of a product with cols_operand
    __device__ static __forceinline__ bf16x8 rows_in_c_order(const Lane& at, int r0, int t) {
        typedef const __attribute__((address_space(3))) u32x2 lds_u32x2;
        const uint32_t off = (uint32_t)(((r0 / 16) * kBlocksAcross + t / 2) * 1024);
        const u32x2 a = *(lds_u32x2*)(at.order[2 * (t & 1)] + off), b = *(lds_u32x2*)(at.order[2 * (t & 1) + 1] + off);
        return as_bf16x8(u32x4{a.x, a.y, b.x, b.y});
    }
    // A operand of the transposed tile: rows = columns d0 .. d0+31 of the tile (d0 a multiple of 32), k = tile rows
    // k0 .. k0+15 (k0 a multiple of 16) in the order 4h + {0..3}, 8 + 4h + {0..3}
    __device__ static __forceinline__ bf16x8 cols_operand(const Lane& at, int tile, int k0, int d0) {
        typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
        const uint32_t off = (uint32_t)(tile + ((k0 / 16) * kBlocksAcross + d0 / 32) * 1024);
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at.cols[0] + off));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)(at.cols[1] + off));
        const u32x2 a = __builtin_bit_cast(u32x2, lo), b = __builtin_bit_cast(u32x2, hi);
        return as_bf16x8(u32x4{a.x, a.y, b.x, b.y});
    }
};

// Order of a straight run of matrix instructions and the LDS reads that feed them: `ahead` operands are requested before
// the first product, then one more per product, so that no product waits for the read just issued (left alone, the compiler
// reads each operand right before its use and waits out the latency every time).  READS: LDS instructions per operand.
template <int PRODUCTS, int READS, int AHEAD>
__device__ __forceinline__ void order_products() {
    __builtin_amdgcn_sched_group_barrier(0x100, READS * AHEAD, 0);
#pragma unroll
    for (int i = 0; i < PRODUCTS - AHEAD; ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
        __builtin_amdgcn_sched_group_barrier(0x100, READS, 0);
    }
    __builtin_amdgcn_sched_group_barrier(0x008, AHEAD, 0);
}

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
