// Pieces shared by the LDS-staged GEMM kernels (qkv_prefill.hip, tile_gemm.hip).
#pragma once

#include "qkv_common.h"

namespace tllm {

// Chunk swizzle of LDS row r: the 16-byte chunk c of the row is stored at chunk position c ^ swz(r). Eight consecutive
// rows of one chunk land on the eight chunk positions, and rows r, r + 8 on positions that differ in bit 0.
__device__ __forceinline__ int swz(int r) { return (r ^ (r >> 3)) & 7; }

// Rotary positions of N consecutive rows starting at row g0 (the same in every lane; rows past the last one repeat it), as
// they are when all of them lie in [0, max_ctx), which the return value says. Without a positions tensor one 32-bit division
// finds the first row's place in its sequence and the others follow by counting (a decode batch: every row is one; with a table filled
// row by row 128 rows of 2880 took 18.2 us and take 16.9, 200 rows 20.7 and 18.7, 33 rows of 4096 17.6 and 16.1).
// Otherwise (wrap-around, more than 2^31 rows) the caller fills its table with rope_position(), in
// a rolled loop: the 64-bit divisions inlined per row were 32 KB of code to fetch, executed or not, at about 1 us per 8 KB.
// Read through the scalar cache: positions and offset were written before this kernel started and nothing writes them while
// it runs, and a scalar load does not involve the vector-memory counter the look-ahead loads are waited for with.
template <int N>
__device__ __forceinline__ bool rope_positions_uniform(const RopeArgs& r, const void* any_valid, int64_t g0, int64_t rows, int (&pos)[N]) {
  typedef const int64_t __attribute__((address_space(4))) * const_i64_ptr;
  // branch-free (an absent tensor reads a valid dummy address), so that the values stay in scalar registers
  const_i64_ptr pp = reinterpret_cast<const_i64_ptr>(reinterpret_cast<uintptr_t>(r.positions ? static_cast<const void*>(r.positions) : any_valid));
  const_i64_ptr po = reinterpret_cast<const_i64_ptr>(reinterpret_cast<uintptr_t>(r.offset ? static_cast<const void*>(r.offset) : any_valid));
  const int64_t off_ld = po[0];
  const int64_t off = r.offset ? off_ld : 0;
  const bool counts = rows < (1ll << 31);
  // a sequence longer than the batch is as good as one that ends with it
  const unsigned length = static_cast<unsigned>(r.tokens_per_batch < rows ? r.tokens_per_batch : rows);
  const int64_t start = g0 < rows ? g0 : rows - 1;
  unsigned within = counts ? static_cast<unsigned>(start) % length : 0;
  uint64_t most = 0;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    const int64_t gi = g0 + j < rows ? g0 + j : rows - 1;
    const int64_t ld = pp[r.positions ? gi : 0];
    const uint64_t q = static_cast<uint64_t>(r.positions ? ld : off + static_cast<int64_t>(within));
    if (g0 + j + 1 < rows) within = within + 1 == length ? 0 : within + 1;
    pos[j] = static_cast<int>(q);
    if (q > most) most = q;
  }
  return most < static_cast<uint64_t>(r.max_ctx) && most < (1ull << 31) && (r.positions || counts);
}

// (cos, sin) of frequency f at position p in [0, max_ctx)
template <bool TABLE>
__device__ __forceinline__ float2 rope_cos_sin_at(const RopeArgs& r, const YarnFreqs& fr, int p, int f) {
  float c, s;
  if constexpr (TABLE) {
    const int64_t at = p * r.table_row_stride + f;
    c = r.cos_table[at];
    s = r.sin_table[at];
  } else {
    yarn_cos_sin(p, fr.v[f], r.concentration, &c, &s);
  }
  return make_float2(c, s);
}

// Tiles of 64 x 32 .. 128 x 256 (tile_gemm.hip). QKV + bias + rotary: hidden % 64 == 0, head_dim 64, x and W 16-byte aligned,
// weight below 4 GiB.
int launch_tile_gemm_qkv(const char* what, const QkvArgs& a, const RopeArgs& ra, const YarnFreqs& fr, hipStream_t st);
struct TileSize {
  int bm, bn;
};
// The tile that such a launch takes for `rows` rows, `cols` output columns and K = k, and what the host expects it to take, in ns.
TileSize tile_gemm_pick(int64_t rows, int64_t cols, int64_t k, int64_t* ns);
int64_t tile_gemm_ns(int64_t rows, int64_t cols, int64_t k);

// Whether tllm_qkv_rope_decode_bf16 and tllm_qkv_rope_prefill_bf16 take GEMM tiles for aligned operands of these sizes.
bool qkv_decode_tiles(int64_t rows, int64_t hidden, int heads, int head_dim);
bool qkv_prefill_tiles(int64_t rows, int64_t hidden, int heads, int head_dim);

}  // namespace tllm
