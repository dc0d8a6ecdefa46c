// Decode-size attention out-projection with bias and residual:  out[r, n] = sum_k x[r, k] * W[n, k] + b[n] + res[r, n]
// (out_residual_decode_forward, triton_kernels.py:1470-1517; split-K kernel :1340-1416 + reduce :1419-1467).
// One launch, no partial-sum workspace; `out` may be the residual buffer itself, as in the reference.
//
//   out_decode_r8_kernel    (out_decode_r8.hip)  in_dim == 4096, out_dim % 12 == 0 (gpt-oss: [2880, 4096]), up to 8 rows
//   out_decode_r32_kernel   (out_decode_r32.hip) the same shape, more rows in chunks of 32
//                           both: bf16 or fp8 weight, weight-streaming through LDS, twelve output features per workgroup
//   out_decode_general_kernel  (decode_general.hip)  any other in_dim % 32 == 0
//   tile_gemm_kernel        (tile_gemm.hip) a bf16 weight and more rows than out_decode_tiles says
//   out_generic_kernel      anything else: one wavefront per (row, feature) dot product.
//
// W8: fp8 (OCP e4m3) weight with one fp32 scale per output row, as the reference's ATTN_FP8 option
// (triton_kernels.py:1385-1408); the values are widened to bf16 (exact) on their way into LDS and the row scale
// multiplies the finished sum.
#include "out_common.h"
#include "qkv_prefill.h"

namespace tllm {

// Any shape: one wavefront per (row, feature); 2-byte loads, shuffle reduction.
__global__ __launch_bounds__(256) void out_generic_kernel(OutArgs a) {
  const int lane = threadIdx.x & 63;
  const int64_t n = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  const int64_t r = blockIdx.y;
  if (n >= a.out_dim) return;
  const bf16* xrow = a.x + r * a.in_dim;
  float s = 0.f;
  if (a.w_scale) {
    const unsigned char* wrow = reinterpret_cast<const unsigned char*>(a.W) + n * a.in_dim;
    for (int k = lane; k < a.in_dim; k += 64) {
      typedef __attribute__((__vector_size__(2 * sizeof(float)))) float f32x2;
      const f32x2 w = __builtin_amdgcn_cvt_pk_f32_fp8(static_cast<int>(wrow[k]), false);
      s = fmaf(static_cast<float>(xrow[k]), w[0], s);
    }
    s = wave_sum(s) * a.w_scale[n];
  } else {
    const bf16* wrow = reinterpret_cast<const bf16*>(a.W) + n * a.in_dim;
    for (int k = lane; k < a.in_dim; k += 64) s = fmaf(static_cast<float>(xrow[k]), static_cast<float>(wrow[k]), s);
    s = wave_sum(s);
  }
  if (lane != 0) return;
  if (a.bias) s += static_cast<float>(a.bias[n]);
  if (a.res) s += static_cast<float>(a.res[r * a.res_rs + n]);
  a.out[r * a.out_rs + n] = static_cast<bf16>(s);
}

// From where on GEMM tiles are ahead, us, decode kernel / tiles. The kernel for 4096 wide inputs reads its weight once for up to 128 rows in
// chunks that follow each other, which is what it takes: [4096, 2880] 72 rows 12.2 / 13.2, 80 12.8 / 13.2, 96 14.5 / 13.8, 128 17.3 / 15.1, 192
// 27.8 / 16.3, 400 56.9 / 19.6. Narrower outputs leave it as many CUs as it has workgroups of twelve columns, and each its own share of the
// memory: 1536 columns 96 rows 12.3 / 13.2, 128 15.1 / 15.4, 144 15.1 / 12.8; 2304 columns 96 rows 13.4 / 13.5, 144 17.5 / 13.1. More than 256
// workgroups take two rounds: 4032 columns 40 rows 16.0 / 14.5, 96 rows 25.0 / 14.1.
// Any other width, as in qkv_decode_tiles: of 420 points at widths of 512 - 6144, 512 - 5120 columns and 16 - 400 rows 397 within 3 % of the
// better one and none slower than before: [4096, 4096] 64 rows 17.9 / 17.0, 128 rows 34.8 / 16.5, 6144 x 5120 128 rows 93 / 30, 2048 x 2048 128
// rows 10.2 / 9.6, and by the general kernel 1024 x 2880 64 rows 6.3 / 7.2, 2048 x 1024 192 rows 8.6 / 9.7.
bool out_decode_tiles(int64_t rows, int64_t in_dim, int64_t out_dim) {
  if (out_dim % 16 || in_dim % 64 || rows <= 32) return false;
  if (in_dim == 4096 && out_dim % 12 == 0) return rows > (out_dim > 12 * 256 ? 32 : out_dim > 2560 ? 80 : 128);
  const int64_t chunks = (rows + 15) / 16;
  return tile_gemm_ns(rows, out_dim, in_dim) <= decode_general_ns(out_dim / 16 * chunks, in_dim);
}

}  // namespace tllm

using namespace tllm;

extern "C" int tllm_out_gemm_tile(int64_t rows, int64_t in_dim, int64_t out_dim) {
  if (rows < 1 || in_dim < 1 || out_dim < 1 || !out_decode_tiles(rows, in_dim, out_dim)) return 0;
  int64_t ns;
  const TileSize t = tile_gemm_pick(rows, out_dim, in_dim, &ns);
  return t.bm << 16 | t.bn;
}


extern "C" int tllm_out_residual_decode_bf16(const void* x, const void* W, const float* w_scale, const void* bias, const void* residual,
                                             void* out, int64_t res_row_stride, int64_t out_row_stride, int64_t rows, int64_t in_dim,
                                             int64_t out_dim, void* stream) {
  TLLM_REQUIRE(rows >= 0 && in_dim >= 1 && out_dim >= 1, TLLM_E_SHAPE, "out_residual_decode: rows %lld, in_dim %lld, out_dim %lld",
               (long long)rows, (long long)in_dim, (long long)out_dim);
  TLLM_REQUIRE(in_dim < (1ll << 31) && out_dim < (1ll << 31) && in_dim * out_dim < (1ll << 40), TLLM_E_SHAPE,
               "out_residual_decode: weight too large");
  if (rows == 0) return TLLM_OK;
  TLLM_REQUIRE(x && W && out, TLLM_E_ARG, "out_residual_decode: x, W and out must not be NULL");
  TLLM_REQUIRE(out_row_stride >= out_dim && (residual == nullptr || res_row_stride >= out_dim), TLLM_E_ARG,
               "out_residual_decode: row strides must be >= out_dim");
  TLLM_REQUIRE(w_scale == nullptr || reinterpret_cast<uintptr_t>(w_scale) % 4 == 0, TLLM_E_ALIGN, "out_residual_decode: w_scale alignment");
  OutArgs a;
  a.x = (const bf16*)x;
  a.W = W;
  a.w_scale = w_scale;
  a.bias = (const bf16*)bias;
  a.res = (const bf16*)residual;
  a.out = (bf16*)out;
  a.res_rs = res_row_stride;
  a.out_rs = out_row_stride;
  a.rows = rows;
  a.in_dim = (int)in_dim;
  a.out_dim = (int)out_dim;
  hipStream_t st = static_cast<hipStream_t>(stream);
  // (in as many rows as the decode kernels take)
  const bool wide = in_dim == 4096 && out_dim % 12 == 0 && out_dim * in_dim < (1ll << 31);
  if (!w_scale && rows <= (wide ? 32ll : 16ll) * 65535 && out_decode_tiles(rows, in_dim, out_dim) && linear_fits_tiles(x, W, rows, in_dim, out_dim))
    return launch_tile_gemm_out("out_residual_decode", a, st);
  if (wide && aligned16(x) && aligned16(W)) {
    TLLM_REQUIRE((rows + 31) / 32 <= 65535, TLLM_E_SHAPE, "out_residual_decode: rows %lld too many for the decode kernel", (long long)rows);
    if (rows <= 8) launch_out_decode_r8(dim3((unsigned)(out_dim / 12)), st, a);
    else launch_out_decode_r32(st, a);
    return check_launch("out_residual_decode");
  }
  // [4096, 4096] weight, 8 rows: 7.1 us; out_generic_kernel 89.7 (it reads the weight once per row, two bytes a lane)
  if (in_dim % 32 == 0 && aligned16(x) && aligned16(W)) return launch_out_decode_general("out_residual_decode", a, st);
  TLLM_REQUIRE(rows <= 65535, TLLM_E_SHAPE, "out_residual_decode: rows %lld too many for the generic kernel", (long long)rows);
  hipLaunchKernelGGL(out_generic_kernel, dim3((unsigned)((out_dim + 3) / 4), (unsigned)rows), dim3(256), 0, st, a);
  return check_launch("out_residual_decode(generic)");
}
