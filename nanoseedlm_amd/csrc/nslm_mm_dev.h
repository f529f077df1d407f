// nslm_mm_dev.h - what the GEMM sources share: the launch arguments, BF16 packing, and the launcher of the kernel for few tokens.
#pragma once
#include <type_traits>

#include "nslm_mv_dev.h"

namespace nslm {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));

#define OUT_BF16 2   // f32out: the results as BF16 bits (y is uint16_t [][ys])
struct MmArgs {
    int K, R, T, xs, ys, xdiv, add, f32out;
    int least, most;     // grouped: a tile of up to `least` pairs, or of more than `most`, is another launch's;
    int paired;          // so is, beside k_mm_wide, a tile that joins one of k_mm_wide's (Join)
    const WSlice* ws2;   // grouped launches of two matrices over the same tiles (grid.z = 2): the second slice table ..
    float* y2;           // .. and its output
    uint16_t* a16;       // non-null: a workgroup's weight rows are gate rows (ws) and the same rows of up (ws2), half and half, and what
                         // it stores is their SwiGLU as BF16 bits [pair][ys] (the two GEMMs and the SwiGLU + pack pass in one launch)
};

__device__ __forceinline__ uint32_t cvt_pk_bf16(float lo, float hi) {   // v_cvt_pk_bf16_f32: both round to nearest even
    const f32x2 v = {lo, hi};
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

template <int FMT>
constexpr bool seed_fmt() { return FMT == MF_SEED4P4 || FMT == MF_SEED4; }
template <int FMT>
constexpr int seed_p() { return FMT == MF_SEED4 ? 3 : 4; }
template <int FMT>
constexpr int mm_tab_words() { return seed_fmt<FMT>() ? sum_tab_words<seed_p<FMT>()>() : 1; }
// a sum of products with the weights, scaled as the format has them
template <int FMT>
__device__ __forceinline__ float mm_scale(float v, int eb) { return seed_fmt<FMT>() ? sums_scale(v, eb) : v; }

// a kernel that asks for more dynamic LDS than the default limit has the limit raised to what it needs, once (the kernel is a
// template argument so that every kernel has its own "once": kernels of one signature share a pointer type)
template <auto K>
void allow_big_lds(size_t bytes) {
    static const hipError_t once = bytes > 48 * 1024 ? hipFuncSetAttribute((const void*) K, hipFuncAttributeMaxDynamicSharedMemorySize, (int) bytes)
                                                     : hipSuccess;
    (void) once;
}

// 16-byte slot s of row r of a [rows][64] BF16 tile in LDS holds piece s ^ x_swizzle(r).  A 16-byte read serves 16 lanes at once, which have to reach
// all 64 banks: lanes 0-3, 12-15, 20-23 and 24-27, then 4-11, 16-19 and 28-31, and the same of the upper half (found by timing lane patterns).  With
// 32 rows and two pieces a read (v_mfma_f32_32x32x16) that is x_swizzle; with 16 rows and four (16x16x32) x_swizzle16: 4.8 clocks a read, 8.2 with
// x_swizzle there and 16.2 with none.
__device__ __forceinline__ int x_swizzle(int row) { return ((row >> 1) & 7) ^ ((row & 1) << 2); }
__device__ __forceinline__ int x_swizzle16(int row) { return ((row >> 3) & 1) * 6 + ((row >> 1) & 1); }

// the kernel for few tokens a matrix (nslm_mm_rows.hip); packed: X holds BF16 bits, else f32
bool mm_rows_better(int fmt, int R, int T, bool packed);
void mm_rows_dense(hipStream_t st, int fmt, const MmArgs& a, const WSlice& w, const void* X, bool packed, float* Y);
void mm_rows_grouped(hipStream_t st, int fmt, const MmArgs& a, const WSlice* ws, const void* X, bool packed, float* Y, const int32_t* perm,
                     const MmTile* tiles, const int32_t* ntiles, int grid_tiles, int tile_rows);

void mm_wide_grouped(hipStream_t st, int fmt, const MmArgs& a, const WSlice* ws, const uint16_t* X, float* Y, const int32_t* perm, const MmTile* tiles,
                     const int32_t* ntiles, int grid_tiles);

}   // namespace nslm
