// Argument block shared by the decode out-projection kernels (out_decode.hip, out_decode_r8.hip, out_decode_r32.hip, decode_general.hip, tile_gemm.hip).
#pragma once
#include "common.h"

namespace tllm {

struct OutArgs {
  const bf16* x;          // [rows, in_dim]
  const void* W;          // [out_dim, in_dim] bf16, or fp8 bytes when w_scale != null
  const float* w_scale;   // [out_dim] or null
  const bf16* bias;       // [out_dim] or null
  const bf16* res;        // [rows, out_dim] with row stride res_rs, or null
  bf16* out;              // [rows, out_dim] with row stride out_rs
  int64_t res_rs, out_rs;
  int64_t rows;
  int in_dim, out_dim;
};

// in_dim 4096, out_dim % 12 == 0, rows <= 8, bf16 weight or (a.w_scale != null) fp8; grid = (out_dim / 12)
void launch_out_decode_r8(dim3 grid, hipStream_t st, const OutArgs& a);

// in_dim 4096, out_dim % 12 == 0, bf16 or fp8 weight, up to 65535 x 32 rows in chunks of up to 32
void launch_out_decode_r32(hipStream_t st, const OutArgs& a);

// any in_dim % 32 == 0 and out_dim, bf16 or fp8 weight, any rows in chunks of 8 or 16; x and W 16-byte aligned
int launch_out_decode_general(const char* what, const OutArgs& a, hipStream_t st);

// GEMM tiles (tile_gemm.hip), bf16 weight: whether they take these operands, and the launch
bool linear_fits_tiles(const void* x, const void* W, int64_t rows, int64_t in_dim, int64_t out_dim);
int launch_tile_gemm_out(const char* what, const OutArgs& a, hipStream_t st);

// Whether tllm_out_residual_decode_bf16 takes them for aligned operands of these sizes and a bf16 weight (out_decode.hip)
bool out_decode_tiles(int64_t rows, int64_t in_dim, int64_t out_dim);

}  // namespace tllm
