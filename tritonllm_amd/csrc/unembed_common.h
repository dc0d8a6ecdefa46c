// Shared by the decode-size unembedding kernels (unembed.hip, unembed_tiles.hip).
#pragma once

#include "common.h"

namespace tllm {

struct UnembedArgs {
  const bf16* x;          // [rows, hidden]
  const void* W;          // [vocab, hidden] bf16, or fp8 bytes when w_scale != null
  const float* w_scale;   // [vocab] or null
  bf16* logits;           // [rows, vocab] with row stride ld (logits form)
  int64_t ld;
  float* part_max;        // [gridDim.y][gridDim.x * UNW][XR] (argmax form)
  int* part_idx;
  int64_t rows;
  int hidden, vocab;
  int pair_stores;        // the logits rows allow 4-byte stores at even columns
};

constexpr int kUnembedGrid = 256;      // one workgroup per CU

// Logits of up to 128 rows per pass over the weight (unembed_tiles.hip): which calls it can take, and the launch.
bool unembed_tiles_fit(int64_t rows, bool w8, int64_t hidden, int64_t vocab);
int unembed_tile_units(int64_t rows, bool w8, int64_t vocab);          // of its widest tile
int launch_unembed_tiles(const char* who, const UnembedArgs& a, bool w8, hipStream_t st);

}  // namespace tllm
