// Decode-size projections at shapes other than gpt-oss's, over the stream of decode_general_stream.h: a workgroup owns
// sixteen weight rows and up to XR activation rows, four wavefronts stream, a fifth one loads what the epilogue needs
// while they do (bias, residual, row scales, rotary position and cos / sin), adds the partial tiles and stores.
//
//   qkv_decode_general_kernel  QKV + bias + rotary, any hidden % 32 == 0, head_dim % 16 == 0 (the reference's decode kernel
//                              is generic over both, triton_kernels.py:1127-1158, 927-940)
//   out_decode_general_kernel  out-projection + bias + residual, any in_dim % 32 == 0 (triton_kernels.py:1340-1467)
//
// HBM-bound: 8 rows, [4096, 4096] weight 7.1 us = 4.7 TB/s, of which 1.6 us are the launch (a wavefront per dot product:
// 89.7 us); QKV at hidden 4096, 80 heads of 64 11.0 us = 3.8 TB/s (14.7 before), fp8 weight 8.0 (13.5). Above 8 rows the
// sixteen-row form: its activations are half of what a workgroup reads, from the L2s.
#include "decode_general_stream.h"
#include "out_common.h"
#include "qkv_common.h"

namespace tllm {

// Rows [8 piece, 8 piece + 8) of a head and their rotation partners half = head_dim / 2 further on; tile row 4 qd + i is
// dim 8 piece + 2 qd + (i & 1), plus half when i >= 2, so that a lane's four sums are two complete (lo, hi) pairs.
template <int XR, bool W8>
__global__ __launch_bounds__(320) void qkv_decode_general_kernel(QkvArgs a, RopeArgs ra, YarnFreqs fr) {
  using S = DecodeGeneralStream<XR, W8>;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int half = a.head_dim >> 1, pieces = half >> 3;
  const int head = blockIdx.x / pieces, piece = blockIdx.x - head * pieces;
  const int64_t row0 = static_cast<int64_t>(blockIdx.y) * XR;
  const int nvalid = static_cast<int>(a.rows - row0 < XR ? a.rows - row0 : XR);
  if (wave < S::NS) {
    const unsigned char* wbase = reinterpret_cast<const unsigned char*>(a.W) + static_cast<int64_t>(head) * a.head_dim * a.hidden * (W8 ? 1 : 2);
    S::run(smem, wave, lane, reinterpret_cast<const unsigned char*>(a.x + row0 * a.hidden), nvalid, wbase,
           [&](int i) { return 8 * piece + 2 * (i >> 2) + (i & 1) + ((i & 2) ? half : 0); }, a.hidden);
    __syncthreads();
    return;
  }
  const int m = lane & 15, g = lane >> 4;
  const int64_t row = row0 + (m < nvalid ? m : 0);
  const bool rotate = a.has_rope && head < a.n_q_heads + a.n_kv_heads;
  const int d0 = 8 * piece + 2 * g, col = head * a.head_dim + d0;
  bf16* out = qkv_out_ptr(a, qkv_slot(a, ra), row, head) + d0;
  float b[4] = {0.f, 0.f, 0.f, 0.f}, s[4] = {1.f, 1.f, 1.f, 1.f}, c0 = 1.f, s0 = 0.f, c1 = 1.f, s1 = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = col + (i & 1) + ((i & 2) ? half : 0);
    if (a.bias) b[i] = static_cast<float>(a.bias[at]);
    if constexpr (W8) s[i] = a.w_scale[at];
  }
  if (rotate) {
    const int64_t pos = rope_position(ra, row);
    rope_cos_sin(ra, fr, pos, d0, &c0, &s0);
    rope_cos_sin(ra, fr, pos, d0 + 1, &c1, &s1);
  }
  // pinned ahead of the barrier: one wavefront runs alone from there to the stores
  asm volatile("" : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]), "+v"(c0), "+v"(s0), "+v"(c1), "+v"(s1), "+v"(out));
  if constexpr (W8) asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]));
  __syncthreads();
  const f32x4 t = S::sum(smem, lane);
  if (m >= nvalid) return;
  const float lo0 = t[0] * s[0] + b[0], lo1 = t[1] * s[1] + b[1], hi0 = t[2] * s[2] + b[2], hi1 = t[3] * s[3] + b[3];
  bf16x2 lo, hi;
  lo[0] = static_cast<bf16>(rotate ? lo0 * c0 - hi0 * s0 : lo0);
  lo[1] = static_cast<bf16>(rotate ? lo1 * c1 - hi1 * s1 : lo1);
  hi[0] = static_cast<bf16>(rotate ? hi0 * c0 + lo0 * s0 : hi0);
  hi[1] = static_cast<bf16>(rotate ? hi1 * c1 + lo1 * s1 : hi1);
  *reinterpret_cast<bf16x2*>(out) = lo;
  *reinterpret_cast<bf16x2*>(out + half) = hi;
}

template <int XR, bool W8>
__global__ __launch_bounds__(320) void out_decode_general_kernel(OutArgs a, int vec8) {
  using S = DecodeGeneralStream<XR, W8>;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int n0 = blockIdx.x * 16;
  const int64_t row0 = static_cast<int64_t>(blockIdx.y) * XR;
  const int nvalid = static_cast<int>(a.rows - row0 < XR ? a.rows - row0 : XR);
  if (wave < S::NS) {
    const unsigned char* wbase = reinterpret_cast<const unsigned char*>(a.W) + static_cast<int64_t>(n0) * a.in_dim * (W8 ? 1 : 2);
    const int last = a.out_dim - 1 - n0;
    S::run(smem, wave, lane, reinterpret_cast<const unsigned char*>(a.x + row0 * a.in_dim), nvalid, wbase,
           [&](int i) { return i < last ? i : last; }, a.in_dim);
    __syncthreads();
    return;
  }
  const int m = lane & 15, g = lane >> 4;
  const int64_t row = row0 + (m < nvalid ? m : 0);
  const int feat = n0 + 4 * g, nfeat = a.out_dim - feat < 4 ? a.out_dim - feat : 4;   // the lane's four features (none: <= 0)
  float b[4] = {0.f, 0.f, 0.f, 0.f}, r[4] = {0.f, 0.f, 0.f, 0.f}, s[4] = {1.f, 1.f, 1.f, 1.f};
  if (vec8 && nfeat == 4) {
    if (a.bias) {
      const bf16x4 v = *reinterpret_cast<const bf16x4*>(a.bias + feat);
#pragma unroll
      for (int i = 0; i < 4; ++i) b[i] = static_cast<float>(v[i]);
    }
    if (a.res) {
      const bf16x4 v = *reinterpret_cast<const bf16x4*>(a.res + row * a.res_rs + feat);
#pragma unroll
      for (int i = 0; i < 4; ++i) r[i] = static_cast<float>(v[i]);
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if (i >= nfeat) continue;
      if (a.bias) b[i] = static_cast<float>(a.bias[feat + i]);
      if (a.res) r[i] = static_cast<float>(a.res[row * a.res_rs + feat + i]);
    }
  }
  if constexpr (W8) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < nfeat) s[i] = a.w_scale[feat + i];
    asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]));
  }
  asm volatile("" : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]), "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]));
  __syncthreads();
  const f32x4 t = S::sum(smem, lane);
  if (m >= nvalid || nfeat <= 0) return;
  bf16* out = a.out + row * a.out_rs + feat;
  bf16x4 o;
#pragma unroll
  for (int i = 0; i < 4; ++i) o[i] = static_cast<bf16>(t[i] * s[i] + b[i] + r[i]);
  if (vec8 && nfeat == 4) {
    *reinterpret_cast<bf16x4*>(out) = o;
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (i < nfeat) out[i] = o[i];
  }
}

namespace {
template <auto kernel, class... Args>
int launch(const char* what, int lds, unsigned gx, int64_t gy, hipStream_t st, const Args&... args) {
  TLLM_REQUIRE(gy <= 65535, TLLM_E_SHAPE, "%s: too many rows for the decode kernel", what);
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> done{0};
    hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds, done);
    TLLM_REQUIRE(e == hipSuccess, TLLM_E_LAUNCH, "%s: cannot raise LDS limit: %s", what, hipGetErrorString(e));
  }
  hipLaunchKernelGGL(kernel, dim3(gx, (unsigned)gy), dim3(320), (size_t)lds, st, args...);
  return check_launch(what);
}
}  // namespace

int launch_qkv_decode_general(const char* what, const QkvArgs& a, const RopeArgs& ra, const YarnFreqs& fr, hipStream_t st) {
  const unsigned gx = (unsigned)((a.n_q_heads + 2 * a.n_kv_heads) * (a.head_dim / 16));
  const bool few = a.rows <= 8;
  const int64_t gy = few ? 1 : (a.rows + 15) / 16;
  if (a.w_scale)
    return few ? launch<qkv_decode_general_kernel<8, true>>(what, DecodeGeneralStream<8, true>::LDS, gx, gy, st, a, ra, fr)
               : launch<qkv_decode_general_kernel<16, true>>(what, DecodeGeneralStream<16, true>::LDS, gx, gy, st, a, ra, fr);
  return few ? launch<qkv_decode_general_kernel<8, false>>(what, DecodeGeneralStream<8, false>::LDS, gx, gy, st, a, ra, fr)
             : launch<qkv_decode_general_kernel<16, false>>(what, DecodeGeneralStream<16, false>::LDS, gx, gy, st, a, ra, fr);
}

int launch_out_decode_general(const char* what, const OutArgs& a, hipStream_t st) {
  auto al8 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 8 == 0; };
  const int vec8 = al8(a.out) && a.out_rs % 4 == 0 && (a.res == nullptr || (al8(a.res) && a.res_rs % 4 == 0)) && (a.bias == nullptr || al8(a.bias));
  const unsigned gx = (unsigned)((a.out_dim + 15) / 16);
  const bool few = a.rows <= 8;
  const int64_t gy = few ? 1 : (a.rows + 15) / 16;
  if (a.w_scale)
    return few ? launch<out_decode_general_kernel<8, true>>(what, DecodeGeneralStream<8, true>::LDS, gx, gy, st, a, vec8)
               : launch<out_decode_general_kernel<16, true>>(what, DecodeGeneralStream<16, true>::LDS, gx, gy, st, a, vec8);
  return few ? launch<out_decode_general_kernel<8, false>>(what, DecodeGeneralStream<8, false>::LDS, gx, gy, st, a, vec8)
             : launch<out_decode_general_kernel<16, false>>(what, DecodeGeneralStream<16, false>::LDS, gx, gy, st, a, vec8);
}

}  // namespace tllm
