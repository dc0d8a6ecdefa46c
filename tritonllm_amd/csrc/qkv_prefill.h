// Pieces shared by the LDS-staged GEMM kernels (qkv_prefill.hip, tile_gemm.hip).
#pragma once

#include "qkv_common.h"

namespace tllm {

// Chunk swizzle of LDS row r: the 16-byte chunk c of the row is stored at chunk position c ^ swz(r). Eight consecutive
// rows of one chunk land on the eight chunk positions, and rows r, r + 8 on positions that differ in bit 0.
__device__ __forceinline__ int swz(int r) { return (r ^ (r >> 3)) & 7; }

// Rotary positions of N consecutive rows starting at row g0 (the same in every lane; rows past the last one get a position that
// some row has), as they are when all of them lie in [0, max_ctx), which the return value says. What is executed here is on every
// launch's way, about 4 ns an instruction: 32-bit arithmetic, one load for a whole run of positions, and the division only where
// there are several sequences (97 rows of 2880 x 80 heads, us: from a positions tensor 15.15, from an offset 15.2, three sequences 15.1;
// with 64-bit values and a clamp and a load for each row 15.2, 15.2 and, its table filled row by row, 16.6; counting in 64 bits with the
// division ahead of all of them 15.7, 15.5 and 15.5. 512 x 12 heads 5.69, 5.63, 5.72; 5.73, 5.71, 7.21; 6.10, 6.00, 6.01).
// Otherwise (wrap-around, 2^28 rows and more) the caller fills its table with rope_position(), in
// a rolled loop: the 64-bit divisions inlined per row were 32 KB of code to fetch, executed or not, at about 1 us per 8 KB.
// Read through the scalar cache: positions and offset were written before this kernel started and nothing writes them while
// it runs, and a scalar load does not involve the vector-memory counter the look-ahead loads are waited for with.
template <int N>
__device__ __forceinline__ bool rope_positions_uniform(const RopeArgs& r, int64_t g0, int64_t rows, int (&pos)[N]) {
  typedef const int64_t __attribute__((address_space(4))) * const_i64_ptr;
#pragma unroll
  for (int j = 0; j < N; ++j) pos[j] = 0;
  if (rows >= (1ll << 28)) return false;
  const unsigned limit = r.max_ctx < (1ll << 31) ? static_cast<unsigned>(r.max_ctx) : 1u << 31;
  const unsigned last = static_cast<unsigned>(rows) - 1, first = g0 < rows ? static_cast<unsigned>(g0) : last;
  if (r.positions) {
    const const_i64_ptr pp = reinterpret_cast<const_i64_ptr>(reinterpret_cast<uintptr_t>(r.positions));
    int64_t p[N];
    if (last - first >= N - 1) {                               // one run of N positions
#pragma unroll
      for (int j = 0; j < N; ++j) p[j] = (pp + first)[j];
    } else {
#pragma unroll
      for (int j = 0; j < N; ++j) p[j] = pp[first + j < last ? first + j : last];
    }
    unsigned high = 0, most = 0;
#pragma unroll
    for (int j = 0; j < N; ++j) {
      pos[j] = static_cast<int>(p[j]);
      high |= static_cast<unsigned>(static_cast<uint64_t>(p[j]) >> 32);
      most = static_cast<unsigned>(p[j]) > most ? static_cast<unsigned>(p[j]) : most;
    }
    return high == 0 && most < limit;
  }
  // Without a positions tensor one 32-bit division finds the first row's place in its sequence and the others follow by counting.
  const int64_t off = r.offset ? *reinterpret_cast<const_i64_ptr>(reinterpret_cast<uintptr_t>(r.offset)) : 0;
  const bool several = rows > r.tokens_per_batch;
  const unsigned length = several ? static_cast<unsigned>(r.tokens_per_batch) : 1u << 31;
  const unsigned within = several ? first % length : first;
  // the last place that one of these rows has; where a sequence ends among them, its end
  const unsigned ahead = last - first < N - 1 ? last - first : N - 1, end = within + ahead < length ? within + ahead : length - 1;
  unsigned at = within;
#pragma unroll
  for (int j = 0; j < N; ++j) {
    pos[j] = static_cast<int>(static_cast<unsigned>(off) + (at < end ? at : end));
    at = at + 1 == length ? 0 : at + 1;
  }
  return off >= 0 && static_cast<uint64_t>(off) + end < limit;
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
