// Decode-size projections at shapes other than gpt-oss's, over the stream of decode_general_stream.h: a workgroup owns
// sixteen weight rows and up to XR activation rows, up to four wavefronts stream, one more loads what the epilogue needs
// while they do (bias, residual, row scales, rotary position and cos / sin), adds the partial tiles and stores.
//
//   qkv_decode_general_kernel  QKV + bias + rotary, any hidden % 32 == 0, head_dim % 16 == 0 (the reference's decode kernel
//                              is generic over both, triton_kernels.py:1127-1158, 927-940)
//   out_decode_general_kernel  out-projection + bias + residual, any in_dim % 32 == 0 (triton_kernels.py:1340-1467)
//
// HBM-bound: 8 rows, [4096, 4096] weight 7.1 us = 4.7 TB/s, of which 1.6 us are the launch (a wavefront per dot product:
// 89.7 us); QKV at hidden 4096, 80 heads of 64 11.0 us = 3.8 TB/s (14.7 before), fp8 weight 8.0 (13.5). Above 8 rows the
// sixteen-row form: its activations are half of what a workgroup reads, from the L2s, and there are as many workgroups per
// weight row as chunks of rows (streams below).
#include "decode_general_stream.h"
#include "out_common.h"
#include "qkv_common.h"

namespace tllm {

// Rows [8 piece, 8 piece + 8) of a head and their rotation partners half = head_dim / 2 further on; tile row 4 qd + i is
// dim 8 piece + 2 qd + (i & 1), plus half when i >= 2, so that a lane's four sums are two complete (lo, hi) pairs.
template <int XR, bool W8, int NS>
__global__ __launch_bounds__(64 * (NS + 1)) void qkv_decode_general_kernel(QkvArgs a, RopeArgs ra, YarnFreqs fr) {
  using S = DecodeGeneralStream<XR, W8, NS>;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int half = a.head_dim >> 1, pieces = half >> 3;
  const int head = blockIdx.x / pieces, piece = blockIdx.x - head * pieces;
  const int64_t row0 = static_cast<int64_t>(blockIdx.y) * XR;
  const int nvalid = static_cast<int>(a.rows - row0 < XR ? a.rows - row0 : XR);
  if (wave < NS) {
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
  const f32x4 t = S::sum(smem, lane, a.hidden);
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

template <int XR, bool W8, int NS>
__global__ __launch_bounds__(64 * (NS + 1)) void out_decode_general_kernel(OutArgs a, int vec8) {
  using S = DecodeGeneralStream<XR, W8, NS>;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
  const int n0 = blockIdx.x * 16;
  const int64_t row0 = static_cast<int64_t>(blockIdx.y) * XR;
  const int nvalid = static_cast<int>(a.rows - row0 < XR ? a.rows - row0 : XR);
  if (wave < NS) {
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
  const f32x4 t = S::sum(smem, lane, a.in_dim);
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
// Streaming wavefronts of a workgroup: no more than K has phases for, and four as long as all workgroups are on
// the machine with them. Beyond that fewer, whose LDS lets more workgroups onto a CU (24 KB per wavefront with an fp8 weight:
// one of 96 KB, three of 48, six): a workgroup's fixed time is then somebody else's stream. us, a wavefront per workgroup (the kernel
// before this one), four, two, one; fp8, 80 heads of 64:
//   hidden 1536, 400 rows (8000 workgroups) 61.0 78.4 43.6 37.0   64 rows (1280) 13.8 16.2 11.5 9.3   32 rows (640) 9.9 10.0 6.9 6.9
//   4096, 400 rows 154 138 113 107   64 rows 29.0 24.9 23.0 18.9   32 rows 19.3 15.7 12.5 12.9   12 rows (320) 14.0 10.1 9.3 12.0
//   32 heads, 1536, 32 rows (256) 6.3 4.5 4.8 6.3   150 rows (1280) 13.3 14.8 10.7 9.0
//   bf16, 4096, 24 heads of 128, 32 rows (384) 14.4 13.5 13.5 14.9   64 rows (768) 19.9 18.3 17.7 16.2   12 rows of 80 heads (320) 15.5 12.3 12.7 15.9
// and four wavefronts' LDS where K is one phase (fp8, 256 wide, 400 rows 28.7 before, 57.2, now 14.7). Up to eight rows there are as
// many workgroups as the weight has sixteen rows: four.
template <int XR, bool W8>
int streams(int K, int64_t workgroups) {
  constexpr int KPH = DecodeGeneralStream<XR, W8, 1>::KPH;
  const int most = K > 2 * KPH ? 4 : K > KPH ? 2 : 1;
  if (XR == 8) return most;
  const int fill = workgroups <= (W8 ? 256 : 352) ? 4 : workgroups <= (W8 ? 768 : 512) ? 2 : 1;
  return fill < most ? fill : most;
}

template <class S, auto kernel, int NS, class... Args>
int launch(const char* what, int K, unsigned gx, int64_t gy, hipStream_t st, const Args&... args) {
  TLLM_REQUIRE(gy <= 65535, TLLM_E_SHAPE, "%s: too many rows for the decode kernel", what);
  const int lds = NS * S::wave_lds(K);
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> done{0};
    hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(kernel), lds, done);   // (the larger of the kernel's two sizes)
    TLLM_REQUIRE(e == hipSuccess, TLLM_E_LAUNCH, "%s: cannot raise LDS limit: %s", what, hipGetErrorString(e));
  }
  hipLaunchKernelGGL(kernel, dim3(gx, (unsigned)gy), dim3(64 * (NS + 1)), (size_t)lds, st, args...);
  return check_launch(what);
}

template <int XR, bool W8>
int launch_qkv(const char* what, unsigned gx, int64_t gy, hipStream_t st, const QkvArgs& a, const RopeArgs& ra, const YarnFreqs& fr) {
  switch (streams<XR, W8>(a.hidden, gx * gy)) {
    case 4: return launch<DecodeGeneralStream<XR, W8, 4>, qkv_decode_general_kernel<XR, W8, 4>, 4>(what, a.hidden, gx, gy, st, a, ra, fr);
    case 2: return launch<DecodeGeneralStream<XR, W8, 2>, qkv_decode_general_kernel<XR, W8, 2>, 2>(what, a.hidden, gx, gy, st, a, ra, fr);
    default: return launch<DecodeGeneralStream<XR, W8, 1>, qkv_decode_general_kernel<XR, W8, 1>, 1>(what, a.hidden, gx, gy, st, a, ra, fr);
  }
}

template <int XR, bool W8>
int launch_out(const char* what, unsigned gx, int64_t gy, hipStream_t st, const OutArgs& a, int vec8) {
  switch (streams<XR, W8>(a.in_dim, gx * gy)) {
    case 4: return launch<DecodeGeneralStream<XR, W8, 4>, out_decode_general_kernel<XR, W8, 4>, 4>(what, a.in_dim, gx, gy, st, a, vec8);
    case 2: return launch<DecodeGeneralStream<XR, W8, 2>, out_decode_general_kernel<XR, W8, 2>, 2>(what, a.in_dim, gx, gy, st, a, vec8);
    default: return launch<DecodeGeneralStream<XR, W8, 1>, out_decode_general_kernel<XR, W8, 1>, 1>(what, a.in_dim, gx, gy, st, a, vec8);
  }
}

int64_t chunks_of(int64_t rows) { return rows <= 8 ? 1 : (rows + 15) / 16; }
}  // namespace

// Up to 256 and 512 workgroups 3.3 us and 1.1 / 1.86 ns per element of K, beyond 3.05 us and for each of them 0.41 ns and 0.0045 per
// element: fitted to widths of 64 - 8192, 1 - 144 heads of 64 and 33 - 448 rows.
int64_t decode_general_ns(int64_t workgroups, int64_t K) {
  return workgroups > 512 ? 3050 + workgroups * 41 / 100 + workgroups * K * 45 / 10000 : 3300 + K * (workgroups > 256 ? 186 : 110) / 100;
}

int launch_qkv_decode_general(const char* what, const QkvArgs& a, const RopeArgs& ra, const YarnFreqs& fr, hipStream_t st) {
  const unsigned gx = (unsigned)((a.n_q_heads + 2 * a.n_kv_heads) * (a.head_dim / 16));
  const bool few = a.rows <= 8;
  const int64_t gy = chunks_of(a.rows);
  if (a.w_scale) return few ? launch_qkv<8, true>(what, gx, gy, st, a, ra, fr) : launch_qkv<16, true>(what, gx, gy, st, a, ra, fr);
  return few ? launch_qkv<8, false>(what, gx, gy, st, a, ra, fr) : launch_qkv<16, false>(what, gx, gy, st, a, ra, fr);
}

int launch_out_decode_general(const char* what, const OutArgs& a, hipStream_t st) {
  auto al8 = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 8 == 0; };
  const int vec8 = al8(a.out) && a.out_rs % 4 == 0 && (a.res == nullptr || (al8(a.res) && a.res_rs % 4 == 0)) && (a.bias == nullptr || al8(a.bias));
  const unsigned gx = (unsigned)((a.out_dim + 15) / 16);
  const bool few = a.rows <= 8;
  const int64_t gy = chunks_of(a.rows);
  if (a.w_scale) return few ? launch_out<8, true>(what, gx, gy, st, a, vec8) : launch_out<16, true>(what, gx, gy, st, a, vec8);
  return few ? launch_out<8, false>(what, gx, gy, st, a, vec8) : launch_out<16, false>(what, gx, gy, st, a, vec8);
}

}  // namespace tllm

extern "C" int tllm_decode_general_streams(int64_t rows, int64_t in_dim, int64_t out_dim, int fp8) {
  using namespace tllm;
  if (rows < 1 || in_dim < 1 || in_dim > INT32_MAX || out_dim < 1) return 0;
  const int K = static_cast<int>(in_dim);
  const int64_t workgroups = (out_dim + 15) / 16 * chunks_of(rows);
  if (rows <= 8) return fp8 ? streams<8, true>(K, workgroups) : streams<8, false>(K, workgroups);
  return fp8 ? streams<16, true>(K, workgroups) : streams<16, false>(K, workgroups);
}
