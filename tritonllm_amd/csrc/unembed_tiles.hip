// Logits of more rows than fit the LDS next to the weight stream (unembed.hip): up to 128 batch rows per pass over the
// weight, bf16 or fp8 (one fp32 scale per vocabulary row).
//
//   logits[r, v] = sum_k x[r, k] * W[v, k]
//
// What bounds it is the weight, 1.16 GB at gpt-oss's size, and the kernels for few rows read it once per chunk of 32 rows
// (of 8, for a model too wide for 32 rows in the LDS). Here K is cut into slices of 64 instead, and a slice of the
// activations travels with the weight's: one workgroup of eight wavefronts per CU owns a contiguous run of the vocabulary
// for the whole launch and walks it in tiles of up to 256 vocabulary rows (the run divided evenly: 49 sixteen-row units per
// CU are four tiles of thirteen, not three of sixteen and one of one), and the ring of S stages -- global memory straight
// into LDS, 16-byte chunks XOR-swizzled by row -- runs on across tiles, so that 64-96 KB of the weight are in flight per CU
// from the first instruction to the last. The activations (737 KB at 128 rows) come from the L2, once per tile: a stage is
// 32 KB of weight and 4-16 KB of them, and they take their share of the loads a CU can have in flight, which is what the
// time grows with (tiles of 128: 49 rows 225 us against 219, 128 rows 280 against 261). Wavefronts: four over the
// vocabulary (four units each) x two over the batch rows, on v_mfma_f32_16x16x32_bf16 with the vocabulary on M, so that a
// lane ends up with four consecutive logits of a row. One barrier per stage.
//
// [rows, 2880] x [201088, 2880], us (before: chunks of 32 rows, of 8 where the width is 4096; a read of the weight alone: 174):
//   bf16   33 rows 205 (377)   49 219 (382)   64 228 (386)   96 245 (586)   128 261 (782)   200 510 (1370)
//   fp8    33 rows 138 (240)   49 145 (251)   64 149 (253)   96 179 (372)   128 209 (491)
//   4096 wide, bf16: 9 rows 251 (520)   32 280 (1035)   64 307 (2065)   128 346 (4098)
#include <atomic>

#include "qkv_prefill.h"
#include "unembed_common.h"

namespace tllm {

namespace unembed_tiles {
constexpr int BK = 64, NW = 8, UNITS = 16;      // K slice; wavefronts; sixteen-row units of a tile
constexpr int MAX_RUN = 64;                    // units of a workgroup's run whose fp8 scales the LDS holds

template <int MB, bool W8>                     // MB blocks of sixteen batch rows
struct Shape {
  static_assert(MB % 2 == 0 && MB >= 2 && MB <= 8, "two wavefronts over the batch rows");
  static constexpr int WROW = W8 ? 64 : 128;                 // LDS bytes of a weight row's slice
  static constexpr int WBYTES = UNITS * 16 * WROW, XBYTES = MB * 16 * 128, STAGE = WBYTES + XBYTES;
  static constexpr int TAIL = W8 ? MAX_RUN * 16 * 4 : 0;
  static constexpr int S_FIT = (160 * 1024 - TAIL) / STAGE, S = S_FIT > 8 ? 8 : S_FIT;
  static constexpr int SMEM = S * STAGE + TAIL;
  static constexpr int LW = (W8 ? 1 : 2) * UNITS / NW;                      // loads of 1 KB per wavefront and stage: its unit of the weight ...
  static constexpr int XR = MB * 2, LX = (XR + 7) / 8;       // ... and XR rows of the activations, eight to a load, the last one may be half
  static constexpr int LPW = LW + LX;
  static_assert(S >= 3 && (S - 2) * LPW < 64, "the loads in flight are countable");
};
}  // namespace unembed_tiles

template <int MB, bool W8>
__global__ __launch_bounds__(512) void unembed_tiles_kernel(UnembedArgs a, int chunk_rows) {
  using namespace unembed_tiles;
  typedef Shape<MB, W8> C;
  constexpr int S = C::S, STAGE = C::STAGE, WBYTES = C::WBYTES, WROW = C::WROW, XR = C::XR, LX = C::LX, LW = C::LW, LPW = C::LPW, TB = MB / 2, UB = UNITS / 4;
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 3, wm = wave >> 2, m16 = lane & 15, g = lane >> 4;

  // ---- this workgroup's run of the vocabulary and its tiles
  const int units = (a.vocab + 15) >> 4, nwg = static_cast<int>(gridDim.x), wg = static_cast<int>(blockIdx.x);
  const int u0 = static_cast<int>(static_cast<int64_t>(wg) * units / nwg), u1 = static_cast<int>(static_cast<int64_t>(wg + 1) * units / nwg);
  const int run = u1 - u0;
  if (run == 0) return;                                      // the whole workgroup
  const int ntiles = (run + UNITS - 1) / UNITS, width = (run + ntiles - 1) / ntiles;   // units per tile (the last one may be narrower)
  const int nk = a.hidden / BK, total = ntiles * nk;         // stages of the stream
  const int64_t row0 = static_cast<int64_t>(blockIdx.y) * chunk_rows;
  const int nrows = static_cast<int>(a.rows - row0 < chunk_rows ? a.rows - row0 : chunk_rows);
  const unsigned wpitch = static_cast<unsigned>(a.hidden) * (W8 ? 1 : 2), xpitch = static_cast<unsigned>(a.hidden) * 2;
  const unsigned char* const x_base = reinterpret_cast<const unsigned char*>(a.x) + row0 * a.hidden * 2;
  const unsigned char* const w_base = reinterpret_cast<const unsigned char*>(a.W) + static_cast<int64_t>(u0) * 16 * wpitch;

  // ---- loads. Wavefront w fetches unit w of the tile (one past the tile's width repeats the last one: lines that are on
  // their way already) and rows w * XR .. of the activations (rows past the last one repeat it; never stored). bf16: eight
  // rows of 128 bytes per load, chunk position L % 8 holds chunk (L % 8) ^ swz(row). fp8: sixteen rows of 64 bytes, position
  // L % 4 holds chunk (L % 4) ^ (row / 4).
  unsigned xoff[LX], woff[LW];
#pragma unroll
  for (int j = 0; j < LX; ++j) {
    int r = wave * XR + 8 * j + (lane >> 3);
    const unsigned c = static_cast<unsigned>((lane & 7) ^ swz(r)) * 16u;
    r = r < nrows ? r : nrows - 1;
    xoff[j] = static_cast<unsigned>(r) * xpitch + c;
  }
  const int run_rows = a.vocab - u0 * 16 < run * 16 ? a.vocab - u0 * 16 : run * 16;
  auto weight_offsets = [&](int tile) {
    const int left = run - tile * width, here = left < width ? left : width;
#pragma unroll
    for (int j = 0; j < LW; ++j) {
      constexpr int LU = W8 ? 1 : 2;                         // loads per unit
      const int u = wave * (UNITS / NW) + j / LU, unit = tile * width + (u < here ? u : here - 1);
      const int r = W8 ? lane >> 2 : 8 * (j % LU) + (lane >> 3);
      const unsigned c = (W8 ? static_cast<unsigned>((lane & 3) ^ (r >> 2)) : static_cast<unsigned>((lane & 7) ^ swz(r))) * 16u;
      const int row = unit * 16 + r < run_rows ? unit * 16 + r : run_rows - 1;
      woff[j] = static_cast<unsigned>(row) * wpitch + c;
    }
  };
  int l_tile = 0, l_k = 0, l_slot = 0;                       // load cursor
  weight_offsets(0);
  const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(smem));
  // The next stage of the stream into the next slot. Always the same number of loads: past the end the last stage comes again.
  auto issue = [&]() {
    const unsigned dst = lds0 + l_slot * STAGE;
    const unsigned char* const wb = w_base + static_cast<int64_t>(l_k) * (W8 ? BK : BK * 2);
    const unsigned char* const xb = x_base + static_cast<int64_t>(l_k) * (BK * 2);
#pragma unroll
    for (int j = 0; j < LW; ++j) {
      const unsigned d = dst + wave * (UNITS / NW * 16 * WROW) + j * 1024;
      // a slice of an fp8 row is half a line, so its line is needed again one stage on: no streaming hint
      if constexpr (W8) asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(d), "v"(woff[j]), "s"(wb) : "memory", "m0");
      else asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(d), "v"(woff[j]), "s"(wb) : "memory", "m0");
    }
#pragma unroll
    for (int j = 0; j < LX; ++j) {
      const unsigned d = dst + WBYTES + (wave * XR + 8 * j) * 128;
      if (8 * j + 8 > XR)                                    // known at compile time; every lane is active here, before and after
        asm volatile("s_mov_b32 m0, %0\n\ts_mov_b32 exec_hi, 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 exec_hi, -1" ::"s"(d), "v"(xoff[j]), "s"(xb)
                     : "memory", "m0");
      else
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(d), "v"(xoff[j]), "s"(xb) : "memory", "m0");
    }
    l_slot = l_slot + 1 == S ? 0 : l_slot + 1;
    if (l_k + 1 < nk) {
      ++l_k;
    } else if (l_tile + 1 < ntiles) {
      l_k = 0;
      weight_offsets(++l_tile);
    }
  };

  float* const scales = reinterpret_cast<float*>(smem + S * STAGE);
  if constexpr (W8) {                                        // the run's scales: loaded (and waited for) ahead of the stream
    for (int i = tid; i < run_rows; i += 512) scales[i] = a.w_scale[u0 * 16 + i];
    __syncthreads();
  }
#pragma unroll 1
  for (int s = 0; s < S - 1; ++s) issue();

  // ---- fragments: lane group g supplies chunk 4 kk + gc of both operands' rows (any assignment will do as long as the two
  // agree); under swz() the sixteen lanes that a 128-bit LDS read is served by (0-7 with 32-39, ...) are on different banks.
  const int gc = (g >> 1) | ((g & 1) << 1);
  int fx_o[TB], fw_o[UB];
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) {
    const int r = 16 * (TB * wm + tb) + m16;
    fx_o[tb] = WBYTES + r * 128 + ((gc ^ swz(r)) << 4);
  }
#pragma unroll
  for (int ub = 0; ub < UB; ++ub) {
    if constexpr (W8) fw_o[ub] = (UB * wn + ub) * 1024 + m16 * 64 + (((gc >> 1) ^ (m16 >> 2)) << 4) + (gc & 1) * 8;
    else fw_o[ub] = (UB * wn + ub) * 2048 + m16 * 128 + ((gc ^ swz(m16)) << 4);
  }
  const bool vec4 = reinterpret_cast<uintptr_t>(a.logits) % 8 == 0 && a.ld % 4 == 0;

  int c_slot = 0;
  for (int tile = 0; tile < ntiles; ++tile) {
    f32x4 acc[UB][TB];
#pragma unroll
    for (int ub = 0; ub < UB; ++ub)
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) acc[ub][tb] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int k = 0; k < nk; ++k) {
      // This wavefront's share of the stage has landed (the S - 2 stages behind it may be in flight; stores of the tile
      // before are younger than all of them, which makes the wait longer, never shorter), then everyone's; and everyone has
      // read the slot that the next loads go into.
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((S - 2) * LPW) : "memory");
      const unsigned char* const st = smem + c_slot * STAGE;
      bf16x8 fx[2][TB], fw[2][UB];
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
#pragma unroll
        for (int ub = 0; ub < UB; ++ub) {
          if constexpr (W8) {
            typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned u32x2;
            const u32x2 raw = *reinterpret_cast<const u32x2*>(st + (fw_o[ub] ^ (kk << 5)));
            fw[kk][ub] = fp8x8_to_bf16x8(raw[0], raw[1]);
          } else {
            fw[kk][ub] = *reinterpret_cast<const bf16x8*>(st + (fw_o[ub] ^ (kk << 6)));
          }
        }
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) fx[kk][tb] = *reinterpret_cast<const bf16x8*>(st + (fx_o[tb] ^ (kk << 6)));
      }
      issue();
#pragma unroll
      for (int kk = 0; kk < 2; ++kk)
#pragma unroll
        for (int ub = 0; ub < UB; ++ub)
#pragma unroll
          for (int tb = 0; tb < TB; ++tb) acc[ub][tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[kk][ub], fx[kk][tb], acc[ub][tb], 0, 0, 0);
      c_slot = c_slot + 1 == S ? 0 : c_slot + 1;
    }
    // ---- the tile's logits: lane (batch row m16 of block tb) has vocabulary rows 4 g .. 4 g + 3 of a unit
    const int left = run - tile * width, here = left < width ? left : width;
#pragma unroll
    for (int ub = 0; ub < UB; ++ub) {
      const int unit = UB * wn + ub;
      if (unit >= here) continue;                            // uniform
      const int lv = (tile * width + unit) * 16 + 4 * g;     // in the run
      f32x4 sc = {1.f, 1.f, 1.f, 1.f};
      if constexpr (W8) sc = *reinterpret_cast<const f32x4*>(scales + lv);
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        const int r = 16 * (TB * wm + tb) + m16;
        if (r >= nrows || lv >= run_rows) continue;
        bf16* const dst = a.logits + (row0 + r) * a.ld + (static_cast<int64_t>(u0) * 16 + lv);
        bf16x4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = static_cast<bf16>(W8 ? acc[ub][tb][e] * sc[e] : acc[ub][tb][e]);
        if (vec4 && lv + 4 <= run_rows) {
          *reinterpret_cast<bf16x4*>(dst) = o;
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (lv + e < run_rows) dst[e] = o[e];
        }
      }
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");            // the re-requested last stages land before the LDS is given back
}

namespace {
template <int MB, bool W8>
int launch_one(const char* who, const UnembedArgs& a, int chunk_rows, int chunks, hipStream_t st) {
  typedef unembed_tiles::Shape<MB, W8> C;
  static std::atomic<uint64_t> done{0};
  const hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(unembed_tiles_kernel<MB, W8>), C::SMEM, done);
  TLLM_REQUIRE(e == hipSuccess, TLLM_E_LAUNCH, "%s: cannot raise LDS limit: %s", who, hipGetErrorString(e));
  hipLaunchKernelGGL((unembed_tiles_kernel<MB, W8>), dim3(kUnembedGrid, (unsigned)chunks), dim3(512), C::SMEM, st, a, chunk_rows);
  return check_launch(who);
}
}  // namespace

// hidden % 64 == 0 and 16-byte alignment are the caller's conditions (unembed_check)
bool unembed_tiles_fit(int64_t rows, bool w8, int64_t hidden, int64_t vocab) {
  const int64_t run = (vocab + 15) / 16 / kUnembedGrid + 1;                      // units of the longest run
  return (!w8 || run <= unembed_tiles::MAX_RUN) && run * 16 * hidden * 2 < (1ll << 32) && hidden * 256 < (1ll << 32) && (rows + 127) / 128 <= 65535;
}

int launch_unembed_tiles(const char* who, const UnembedArgs& a, bool w8, hipStream_t st) {
  const int chunks = static_cast<int>((a.rows + 127) / 128);
  const int chunk_rows = static_cast<int>((a.rows + chunks - 1) / chunks);
  const int mb = (chunk_rows + 31) / 32 * 2;
#define TLLM_TILES(MB) \
  if (mb == MB) return w8 ? launch_one<MB, true>(who, a, chunk_rows, chunks, st) : launch_one<MB, false>(who, a, chunk_rows, chunks, st)
  TLLM_TILES(2);
  TLLM_TILES(4);
  TLLM_TILES(6);
  TLLM_TILES(8);
#undef TLLM_TILES
  set_error("%s: no kernel for chunks of %d rows", who, chunk_rows);
  return TLLM_E_SHAPE;
}

}  // namespace tllm
