// Pieces shared by the LDS-staged GEMM kernels (qkv_prefill.hip, tile_gemm.hip).
#pragma once

#include "qkv_common.h"

namespace tllm {

// Chunk swizzle of LDS row r: the 16-byte chunk c of the row is stored at chunk position c ^ swz(r). Eight consecutive
// rows of one chunk land on the eight chunk positions, and rows r, r + 8 on positions that differ in bit 0.
__device__ __forceinline__ int swz(int r) { return (r ^ (r >> 3)) & 7; }

// Unwrapped rotary positions of 16 consecutive rows starting at row g0 (the same in every lane; rows past the last one
// repeat it), read through the scalar cache: positions and offset were written before this kernel started and nothing
// writes them while it runs, and a scalar load does not involve the vector-memory counter the look-ahead loads are
// waited for with. Without a positions tensor the result is offset[0] alone and the caller adds row % tokens_per_batch.
__device__ __forceinline__ void rope_positions_16_uniform(const RopeArgs& r, const void* any_valid, int64_t g0, int64_t rows, int64_t (&pos_even)[8],
                                                          int64_t (&pos_odd)[8]) {
  typedef const int64_t __attribute__((address_space(4))) * const_i64_ptr;
  // branch-free (an absent tensor reads a valid dummy address), so that the sixteen values stay in scalar registers
  const_i64_ptr pp = reinterpret_cast<const_i64_ptr>(reinterpret_cast<uintptr_t>(r.positions ? static_cast<const void*>(r.positions) : any_valid));
  const_i64_ptr po = reinterpret_cast<const_i64_ptr>(reinterpret_cast<uintptr_t>(r.offset ? static_cast<const void*>(r.offset) : any_valid));
  const int64_t off_ld = po[0];
  const int64_t off = r.offset ? off_ld : 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const int64_t gi = g0 + j < rows ? g0 + j : rows - 1;
    const int64_t ld = pp[r.positions ? gi : 0];
    // two arrays: a lane picks row 2 i or 2 i + 1 by a select between them (of one array the compiler makes an
    // indexed access, and the array then lives in scratch memory)
    if (j & 1) pos_odd[j >> 1] = r.positions ? ld : off;
    else pos_even[j >> 1] = r.positions ? ld : off;
  }
}

// Tiles of 64 x 32 .. 128 x 256 (tile_gemm.hip). QKV + bias + rotary: hidden % 64 == 0, head_dim 64, x and W 16-byte aligned,
// weight below 4 GiB.
int launch_tile_gemm_qkv(const char* what, const QkvArgs& a, const RopeArgs& ra, const YarnFreqs& fr, hipStream_t st);
// What the host expects such a launch to take for `rows` rows, `cols` output columns and K = k, in ns.
int64_t tile_gemm_ns(int64_t rows, int64_t cols, int64_t k);

}  // namespace tllm
