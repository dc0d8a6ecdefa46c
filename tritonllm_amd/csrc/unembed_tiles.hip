// Logits of more rows than fit the LDS next to the weight stream (unembed.hip): up to 128 batch rows per pass over the
// weight, bf16 or fp8 (one fp32 scale per vocabulary row).
//
//   logits[r, v] = sum_k x[r, k] * W[v, k]
//
// What bounds it is the weight, 1.16 GB at gpt-oss's size, and the kernels for few rows read it once per chunk of 32 rows
// (of 8, for a model too wide for 32 rows in the LDS). Here K is cut into slices of 64 instead, and a slice of the
// activations travels with the weight's: one workgroup of eight wavefronts per CU owns a contiguous run of the vocabulary
// for the whole launch and walks it in tiles of up to 20 (bf16) or 28 (fp8) units of sixteen vocabulary rows (the run divided
// evenly: 50 units per CU are three tiles of seventeen, not two of twenty and one of ten), and the ring of S stages -- global
// memory straight into LDS, 16-byte chunks XOR-swizzled by row -- runs on across tiles, so that 64-96 KB of the weight are in
// flight per CU from the first instruction to the last. The activations (737 KB at 128 rows) come from the L2, once per tile.
// A CU takes in 28 GB/s of this stream, weight and activations together (fp8 21; 5.5 MB at 49 rows, 6.7 at 128; its loads come back in
// order, the weight's from memory among them), and more bytes take longer if not in proportion (7.4 MB at 49 rows 34 GB/s): few tall tiles, no row
// of either operand that is not needed, the loads of a stage dealt to the wavefronts one by one. Wavefronts: four over the vocabulary x two over the batch rows, on
// v_mfma_f32_16x16x32_bf16 with the vocabulary on M, so that a lane ends up with four consecutive logits of a row. One barrier
// per stage.
//
// [rows, 2880] x [201088, 2880], us (in brackets four tiles of thirteen units whose stages had room and loads for sixteen; in
// chunks of 32 rows, of 8 where the width is 4096; a read of the weight alone: 174):
//   bf16   33 rows 198 (205, 377)   49 200 (218, 382)   64 205 (228, 386)   96 219 (245, 586)   128 240 (262, 782)   200 465 (510, 1370)
//   fp8    33 rows 133 (143, 240)   49 139 (148, 251)   64 144 (153, 253)   96 157 (177, 372)   128 171 - 178 (193 - 205, 491)
//   4096 wide, bf16: 9 rows 262 (257, 520; on another GPU 283 and 288)   32 275 (285, 1035)   49 273 (294)   128 313 (344, 4098)
#include <atomic>

#include "qkv_prefill.h"
#include "unembed_common.h"

namespace tllm {

namespace unembed_tiles {
constexpr int BK = 64, NW = 8;                 // K slice; wavefronts
constexpr int MAX_RUN = 64;                    // units (sixteen vocabulary rows) of a workgroup's run whose fp8 scales the LDS holds
constexpr int LDS = 160 * 1024;

template <int MB, bool W8, int UB>             // MB blocks of sixteen batch rows, up to UB units for each of the four wavefronts over the vocabulary
struct Shape {
  static_assert(MB % 2 == 0 && MB >= 2 && MB <= 8, "two wavefronts over the batch rows");
  static constexpr int WROW = W8 ? 64 : 128, UBYTES = 16 * WROW;   // LDS bytes of a weight row's slice, of a unit's
  static constexpr int XBYTES = MB * 16 * 128, TAIL = W8 ? MAX_RUN * 16 * 4 : 0;
  static constexpr int LU = W8 ? 1 : 2;                      // loads of 1 KB per unit and stage
  static constexpr int LMAX = (4 * UB * LU + MB * 2 + NW - 1) / NW;         // most loads of a wavefront per stage
  // Every wavefront has LMAX loads, the last one of the stage again where there are fewer (the same bytes to the same place). A
  // stage of a narrow fp8 tile is 4 - 24 KB, and the tests and branches around its loads took 2 - 9 % of its time, us with and without:
  // [rows, 2048] x [65000, 2048] 49 rows 34.6 / 33.8, [50257, 2048] 65 rows 36.7 / 35.5, [65000, 768] 64 rows 18.4 / 18.0, one or two units per
  // CU 5 - 9 %; wider tiles (201088 33 rows 135.4 / 139.1) gain nothing, bf16's have twice the bytes.
  static constexpr bool EVEN = W8 && UB <= 4;
  static constexpr int most(int stages) {                    // units of the widest tile of which so many stages fit
    const int fit = ((LDS - TAIL) / stages - XBYTES) / UBYTES;
    return fit < 4 * UB ? fit : 4 * UB;
  }
};
}  // namespace unembed_tiles

// Wait until at most the loads of `STAGES` stages of `cnt` (<= N) loads each are in flight.
template <int N, int STAGES>
__device__ __forceinline__ void wait_stages(int cnt) {
  if constexpr (N == 0) {
    (void)cnt;                                               // (a wavefront without loads)
  } else {
    if (cnt == N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N * STAGES) : "memory");
    else wait_stages<N - 1, STAGES>(cnt);
  }
}

// S stages in the ring; `slots`: units that a stage has room for, the widest tile of the launch.
template <int MB, bool W8, int UB, int S>
__global__ __launch_bounds__(512) void unembed_tiles_kernel(UnembedArgs a, int chunk_rows, int slots) {
  using namespace unembed_tiles;
  typedef Shape<MB, W8, UB> C;
  constexpr int UBYTES = C::UBYTES, LU = C::LU, LMAX = C::LMAX, TB = MB / 2;
  static_assert((S - 2) * LMAX < 64, "the loads in flight are countable");
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wn = wave & 3, wm = wave >> 2, m16 = lane & 15, g = lane >> 4;
  const int wbytes = slots * UBYTES, stage_bytes = wbytes + C::XBYTES;

  // ---- this workgroup's run of the vocabulary and its tiles
  const int units = (a.vocab + 15) >> 4, nwg = static_cast<int>(gridDim.x), wg = static_cast<int>(blockIdx.x);
  const int u0 = static_cast<int>(static_cast<int64_t>(wg) * units / nwg), u1 = static_cast<int>(static_cast<int64_t>(wg + 1) * units / nwg);
  const int run = u1 - u0;
  if (run == 0) return;                                      // the whole workgroup
  const int ntiles = (run + slots - 1) / slots, width = (run + ntiles - 1) / ntiles;   // units per tile (the last one may be narrower)
  const int nk = a.hidden / BK;
  const int64_t row0 = static_cast<int64_t>(blockIdx.y) * chunk_rows;
  const int nrows = static_cast<int>(a.rows - row0 < chunk_rows ? a.rows - row0 : chunk_rows);
  const unsigned wpitch = static_cast<unsigned>(a.hidden) * (W8 ? 1 : 2), xpitch = static_cast<unsigned>(a.hidden) * 2;
  const unsigned char* const x_base = reinterpret_cast<const unsigned char*>(a.x) + row0 * a.hidden * 2;
  const unsigned char* const w_base = reinterpret_cast<const unsigned char*>(a.W) + static_cast<int64_t>(u0) * 16 * wpitch;

  // ---- loads of a stage, dealt to the wavefronts in turn: the units of the tile (in the last, narrower tile the last unit again
  // behind it: lines that are on their way already), then the activations, eight rows to a load (rows past the last one of an
  // eight repeat it; never stored). bf16: eight rows of 128 bytes per load, chunk position L % 8 holds chunk (L % 8) ^ swz(row).
  // fp8: sixteen rows of 64 bytes, position L % 4 holds chunk (L % 4) ^ (row / 4).
  const int w_loads = width * LU, loads = w_loads + (nrows + 7) / 8;
  const int mine = wave < loads ? (loads - wave + NW - 1) / NW : 0;         // this wavefront's (EVEN: LMAX)
  auto load_of = [&](int j) { return C::EVEN && wave + NW * j >= loads ? loads - 1 : wave + NW * j; };
  const int run_rows = a.vocab - u0 * 16 < run * 16 ? a.vocab - u0 * 16 : run * 16;
  unsigned off[LMAX];
  auto offsets = [&](int tile) {
    const int left = run - tile * width, here = left < width ? left : width;
#pragma unroll
    for (int j = 0; j < LMAX; ++j) {
      const int t = load_of(j);
      if (t < w_loads) {
        const int u = t / LU, unit = tile * width + (u < here ? u : here - 1);
        const int r = W8 ? lane >> 2 : 8 * (t % LU) + (lane >> 3);
        const unsigned c = (W8 ? static_cast<unsigned>((lane & 3) ^ (r >> 2)) : static_cast<unsigned>((lane & 7) ^ swz(r))) * 16u;
        const int row = unit * 16 + r < run_rows ? unit * 16 + r : run_rows - 1;
        off[j] = static_cast<unsigned>(row) * wpitch + c;
      } else {
        int r = 8 * (t - w_loads) + (lane >> 3);
        const unsigned c = static_cast<unsigned>((lane & 7) ^ swz(r)) * 16u;
        r = r < nrows ? r : nrows - 1;
        off[j] = static_cast<unsigned>(r) * xpitch + c;
      }
    }
  };
  int l_tile = 0, l_k = 0, l_slot = 0;                       // load cursor
  offsets(0);
  const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(smem));
  // The next stage of the stream into the next slot. Always the same number of loads: past the end the last stage comes again.
  // (The choices sit inside the assembly, so that the schedule around the loads stays one basic block.)
  auto issue = [&]() {
    const unsigned dst = lds0 + l_slot * stage_bytes;
    const unsigned char* const wb = w_base + static_cast<int64_t>(l_k) * (W8 ? BK : BK * 2);
    const unsigned char* const xb = x_base + static_cast<int64_t>(l_k) * (BK * 2);
#pragma unroll
    for (int j = 0; j < LMAX; ++j) {
      const int t = load_of(j);
      const unsigned d = dst + t * 1024 + (t < w_loads ? 0 : wbytes - w_loads * 1024);
      // a slice of an fp8 row is half a line, so its line is needed again one stage on: no streaming hint
      if constexpr (C::EVEN) {
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(d), "v"(off[j]), "s"(t < w_loads ? wb : xb) : "memory", "m0");
      } else if constexpr (W8) {
        asm volatile("s_mov_b32 m0, %0\n\ts_cmp_lt_i32 %3, %4\n\ts_cbranch_scc0 .Lskip%=\n\tglobal_load_lds_dwordx4 %1, %2\n.Lskip%=:" ::"s"(d), "v"(off[j]),
                     "s"(t < w_loads ? wb : xb), "s"(t), "s"(loads)
                     : "memory", "m0", "scc");
      } else {
        asm volatile("s_mov_b32 m0, %0\n\ts_cmp_lt_i32 %4, %5\n\ts_cbranch_scc0 .Lx%=\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_branch .Lskip%=\n.Lx%=:\n\t"
                     "s_cmp_lt_i32 %4, %6\n\ts_cbranch_scc0 .Lskip%=\n\tglobal_load_lds_dwordx4 %1, %3\n.Lskip%=:" ::"s"(d), "v"(off[j]), "s"(wb), "s"(xb), "s"(t),
                     "s"(w_loads), "s"(loads)
                     : "memory", "m0", "scc");
      }
    }
    l_slot = l_slot + 1 == S ? 0 : l_slot + 1;
    if (l_k + 1 < nk) {
      ++l_k;
    } else if (l_tile + 1 < ntiles) {
      l_k = 0;
      offsets(++l_tile);
    }
  };

  float* const scales = reinterpret_cast<float*>(smem + S * stage_bytes);
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
    fx_o[tb] = wbytes + r * 128 + ((gc ^ swz(r)) << 4);
  }
#pragma unroll
  for (int ub = 0; ub < UB; ++ub) {
    const int unit = 4 * ub + wn < width ? 4 * ub + wn : width - 1;          // (past the tile's width: not stored)
    if constexpr (W8) fw_o[ub] = unit * UBYTES + m16 * 64 + (((gc >> 1) ^ (m16 >> 2)) << 4) + (gc & 1) * 8;
    else fw_o[ub] = unit * UBYTES + m16 * 128 + ((gc ^ swz(m16)) << 4);
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
      if constexpr (C::EVEN) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2) * LMAX) : "memory");
      else wait_stages<LMAX, S - 2>(mine);
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
      const unsigned char* const st = smem + c_slot * stage_bytes;
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
      const int unit = 4 * ub + wn;
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
template <int MB, bool W8, int UB, int S>
int launch_one(const char* who, const UnembedArgs& a, int chunk_rows, int chunks, int slots, hipStream_t st) {
  typedef unembed_tiles::Shape<MB, W8, UB> C;
  static std::atomic<uint64_t> done{0};
  const int smem = S * (slots * C::UBYTES + C::XBYTES) + C::TAIL;
  const hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(unembed_tiles_kernel<MB, W8, UB, S>), unembed_tiles::LDS, done);
  TLLM_REQUIRE(e == hipSuccess, TLLM_E_LAUNCH, "%s: cannot raise LDS limit: %s", who, hipGetErrorString(e));
  hipLaunchKernelGGL((unembed_tiles_kernel<MB, W8, UB, S>), dim3(kUnembedGrid, (unsigned)chunks), dim3(512), smem, st, a, chunk_rows, slots);
  return check_launch(who);
}

// As few tiles as possible, since each reads the activations once: of up to 20 units (bf16) or 28 (fp8), and of no more than three
// stages fit the LDS. [rows, 2880] x [201088, 2880], 49 / 128 rows, us: four tiles of thirteen units 206 / 253, three of seventeen
// 200 / 240; fp8 147 / 208 and 143 / 234, two of twenty-five 139 / 178. A kernel for each quarter of those widths, as many stages
// as fit it: units past the tile's width are multiplied as well, and a CU that holds a third of a tile wants more stages on
// their way ([rows, 2880] x [8192, 2880], two units per CU, 49 / 128 rows 34 / 47 -> 20 / 30; 2048 wide, 32000 34 / 41 -> 31 / 35).
template <int MB, bool W8>
int tile_units(int64_t vocab) {
  using unembed_tiles::Shape;
  const int run = static_cast<int>(((vocab + 15) / 16 + kUnembedGrid - 1) / kUnembedGrid);
  constexpr int widest = Shape<MB, W8, W8 ? 7 : 5>::most(3);
  const int tiles = (run + widest - 1) / widest;
  const int slots = (run + tiles - 1) / tiles;
  // fp8: for tiles of 17 - 20 units more than 64 rows leave no room for five stages (from 19, 17 units on at up to 96, 128 rows), and the kernel for 28
  // multiplies eight and more units for nothing. As one tile more: [rows, 2880] x [151936, 2880] 97 rows 147 -> 139 us, 200 rows 285 -> 271, 2048 wide
  // 109 -> 101, 213 -> 198; 96 rows of [234000, 2048] 146 -> 141. One tile stays one (70000 97 rows 72, two 80), and up to 96 rows two stay two
  // (163000 96 rows 135 and 141).
  if (W8 && slots > 16 && slots > Shape<MB, W8, 5>::most(5) && slots <= 20 && tiles > (MB == 8 ? 1 : 2)) return (run + tiles) / (tiles + 1);
  return slots;
}

template <int MB, bool W8>
int launch_shape(const char* who, const UnembedArgs& a, int chunk_rows, int chunks, hipStream_t st) {
  using unembed_tiles::Shape;
  constexpr int BIG = W8 ? 7 : 5;
  const int slots = tile_units<MB, W8>(a.vocab);
  if (slots <= 8) return launch_one<MB, W8, 2, MB <= 4 ? 6 : 5>(who, a, chunk_rows, chunks, slots, st);
  if (slots <= 16) return launch_one<MB, W8, 4, W8 ? (MB == 2 ? 7 : MB == 4 ? 6 : MB == 6 ? 5 : 4) : MB <= 4 ? 4 : 3>(who, a, chunk_rows, chunks, slots, st);
  if constexpr (W8) {
    if (slots <= Shape<MB, W8, 5>::most(5)) return launch_one<MB, W8, 5, 5>(who, a, chunk_rows, chunks, slots, st);
  }
  if (slots <= Shape<MB, W8, BIG>::most(4)) return launch_one<MB, W8, BIG, 4>(who, a, chunk_rows, chunks, slots, st);
  return launch_one<MB, W8, BIG, 3>(who, a, chunk_rows, chunks, slots, st);
}
}  // namespace

// hidden % 64 == 0 and 16-byte alignment are the caller's conditions (unembed_check)
bool unembed_tiles_fit(int64_t rows, bool w8, int64_t hidden, int64_t vocab) {
  const int64_t run = (vocab + 15) / 16 / kUnembedGrid + 1;                      // units of the longest run
  return (!w8 || run <= unembed_tiles::MAX_RUN) && run * 16 * hidden * 2 < (1ll << 32) && hidden * 256 < (1ll << 32) && (rows + 127) / 128 <= 65535;
}

int unembed_tile_units(int64_t rows, bool w8, int64_t vocab) {
  const int64_t chunks = (rows + 127) / 128, mb = ((rows + chunks - 1) / chunks + 31) / 32 * 2;
  if (w8) return mb == 2 ? tile_units<2, true>(vocab) : mb == 4 ? tile_units<4, true>(vocab) : mb == 6 ? tile_units<6, true>(vocab) : tile_units<8, true>(vocab);
  return mb == 2 ? tile_units<2, false>(vocab) : mb == 4 ? tile_units<4, false>(vocab) : mb == 6 ? tile_units<6, false>(vocab) : tile_units<8, false>(vocab);
}

int launch_unembed_tiles(const char* who, const UnembedArgs& a, bool w8, hipStream_t st) {
  const int chunks = static_cast<int>((a.rows + 127) / 128);
  const int chunk_rows = static_cast<int>((a.rows + chunks - 1) / chunks);
  const int mb = (chunk_rows + 31) / 32 * 2;
#define TLLM_TILES(MB) \
  if (mb == MB) return w8 ? launch_shape<MB, true>(who, a, chunk_rows, chunks, st) : launch_shape<MB, false>(who, a, chunk_rows, chunks, st)
  TLLM_TILES(2);
  TLLM_TILES(4);
  TLLM_TILES(6);
  TLLM_TILES(8);
#undef TLLM_TILES
  set_error("%s: no kernel for chunks of %d rows", who, chunk_rows);
  return TLLM_E_SHAPE;
}

}  // namespace tllm
