// MXFP4 -> bf16 expansion of the checkpoint's MoE weights (weights.py:68-117): a block is 16 bytes = 32 fp4 (e2m1)
// values, low nibble first, sharing one e8m0 scale byte:  value = FP4[nibble] * 2^(scale - 127).
// The arithmetic follows the
// reference's torch.ldexp on a bf16 tensor: the product is formed in fp32 and rounded once to bf16 (exact for every
// scale a checkpoint holds; scale bytes >= 255 give inf / nan there and here).
#include "common.h"

namespace tllm {

__device__ __forceinline__ float fp4_value(unsigned nib) {
  // e2m1: 0, 0.5, 1, 1.5, 2, 3, 4, 6 with the sign in bit 3 (weights.py:11-14)
  const unsigned mag = nib & 7u;
  const float m = mag < 2u ? 0.5f * static_cast<float>(mag) : static_cast<float>(2u + (mag & 1u)) * static_cast<float>(1u << ((mag >> 1) - 1u)) * 0.5f;
  return (nib & 8u) ? -m : m;
}

typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned u32x4;

// A lane expands one dword (4 bytes -> 8 values -> one 16-byte store), so that a wave's store covers 1 KB of
// consecutive output and its load 256 consecutive bytes; a work-group takes UNROLL * 256 dwords and each lane issues its
// UNROLL loads before the first conversion.
// gfx950 converts a byte's two values, times a power of two, in one instruction; as long as every nonzero product is a normal
// number (scale bytes 2 .. 252) the result is exact. Lanes whose scale lies outside that range (no checkpoint holds such
// scales) take the fp32 product instead, which covers denormals, inf and nan.
// What bounds it are the writes (1.06 of 1.34 GB; a fill reaches 6.8 TB/s, this 6.0). mlp1 of 32 experts 234 -> 224 us, of three
// 26.0 -> 23.4, 2880 rows of one 7.8 -> 5.0: a table of 256 entries in the LDS stood in the place of the conversion, behind a
// barrier and with its lookups' bank conflicts, and wanted eight dwords per lane to pay for it. With the conversion 1 / 2 / 3 / 4 /
// 8 / 16 dwords per lane take 247 / 224 / 226 / 225 / 239 / 252 us, ordinary stores at eight 245 (239), a contiguous eighth of the
// output per XCD 242, a resident grid 249.
constexpr int MX_UNROLL = 2;
// Blocks of a launch: a grid holds fewer than 2^32 threads, this one 2^31 (16 GB of blocks, 64 GB of output).
constexpr int64_t MX_LAUNCH = 1ll << 30;

__global__ __launch_bounds__(256) void mxfp4_dequant_kernel(const unsigned* __restrict__ blocks, const unsigned char* __restrict__ scales,
                                                            u32x4* __restrict__ out, int64_t n_dwords) {
  const int64_t base = static_cast<int64_t>(blockIdx.x) * (256 * MX_UNROLL) + threadIdx.x;
  unsigned w[MX_UNROLL];
  int e[MX_UNROLL];
#pragma unroll
  for (int u = 0; u < MX_UNROLL; ++u) {
    const int64_t d = base + u * 256;
    w[u] = 0;
    e[u] = 0;
    if (d < n_dwords) {
      w[u] = __builtin_nontemporal_load(blocks + d);
      e[u] = static_cast<int>(scales[d >> 2]) - 127;      // four dwords per block
    }
  }
#pragma unroll
  for (int u = 0; u < MX_UNROLL; ++u) {
    const int64_t d = base + u * 256;
    if (d >= n_dwords) break;
    u32x4 o;
    if (e[u] >= -125 && e[u] <= 125) {
      const float p = __builtin_bit_cast(float, static_cast<unsigned>(e[u] + 127) << 23);
      // byte k gives out[2k] (low nibble) and out[2k+1] (high nibble)
      o[0] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[u], p, 0));
      o[1] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[u], p, 1));
      o[2] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[u], p, 2));
      o[3] = __builtin_bit_cast(unsigned, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w[u], p, 3));
    } else {
      // 2^e as torch.pow(2.0, e) yields it in fp32: denormal below -126, inf above 127
      const float p = e[u] > 127 ? __builtin_inff() : ldexpf(1.0f, e[u]);
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const unsigned byte = (w[u] >> (8 * k)) & 0xffu;
        const bf16 lo = static_cast<bf16>(fp4_value(byte & 15u) * p), hi = static_cast<bf16>(fp4_value(byte >> 4) * p);
        o[k] = static_cast<unsigned>(__builtin_bit_cast(unsigned short, lo)) | (static_cast<unsigned>(__builtin_bit_cast(unsigned short, hi)) << 16);
      }
    }
    __builtin_nontemporal_store(o, out + d);
  }
}

}  // namespace tllm

using namespace tllm;

extern "C" int tllm_mxfp4_dequant_bf16(const void* blocks, const void* scales, void* out, int64_t n_blocks, void* stream) {
  TLLM_REQUIRE(n_blocks >= 0, TLLM_E_ARG, "mxfp4_dequant: n_blocks %lld", (long long)n_blocks);
  if (n_blocks == 0) return TLLM_OK;
  TLLM_REQUIRE(blocks && scales && out, TLLM_E_ARG, "mxfp4_dequant: null pointer");
  TLLM_REQUIRE(aligned16(blocks) && aligned16(out), TLLM_E_ALIGN, "mxfp4_dequant: blocks and out must be 16-byte aligned");
  TLLM_REQUIRE(n_blocks < (1ll << 40), TLLM_E_SHAPE, "mxfp4_dequant: %lld blocks are too many", (long long)n_blocks);
  hipStream_t st = static_cast<hipStream_t>(stream);
  for (int64_t at = 0; at < n_blocks; at += MX_LAUNCH) {
    const int64_t n_dwords = (n_blocks - at < MX_LAUNCH ? n_blocks - at : MX_LAUNCH) * 4;
    hipLaunchKernelGGL(mxfp4_dequant_kernel, dim3((unsigned)((n_dwords + 256 * MX_UNROLL - 1) / (256 * MX_UNROLL))), dim3(256), 0, st,
                       static_cast<const unsigned*>(blocks) + at * 4, static_cast<const unsigned char*>(scales) + at, static_cast<u32x4*>(out) + at * 4, n_dwords);
    const int rc = check_launch("mxfp4_dequant");
    if (rc != TLLM_OK) return rc;
  }
  return TLLM_OK;
}

extern "C" int64_t tllm_mxfp4_launch_threads(int64_t n_blocks) {
  if (n_blocks < 1) return 0;
  const int64_t n_dwords = (n_blocks < MX_LAUNCH ? n_blocks : MX_LAUNCH) * 4;
  return (n_dwords + 256 * MX_UNROLL - 1) / (256 * MX_UNROLL) * 256;
}
