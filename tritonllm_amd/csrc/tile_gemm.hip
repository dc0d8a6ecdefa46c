// GEMM tiles for short prompts and large decode batches: the QKV projection with bias + rotary and the plain projection
// with bias. At 80 heads of 64 and a width of 2880 that is prompts of up to 1536 rows, those for which the larger tiles of
// qkv_prefill.hip would need one more round for little (2049 - 2816, 4097 - 4864, 6145 - 6528, ... rows; qkv_prefill_tiles), and
// decode batches from 113 rows on (qkv_decode_tiles); the plain projection where it is ahead of the library's GEMM, up to
// 2560 rows of [2880, 4096] (linear_in_tiles in host_ops.cpp). With a residual in the epilogue it is the out-projection of decode
// batches from 81 rows on (out_decode_tiles: [4096, 2880] 96 rows 14.5 -> 13.8 us, 128 17.3 -> 15.1, 200 30.6 -> 16.3; [4096, 4096] 128 33.6 -> 16.7).
//
//   D[rows, n] = X[rows, K] . W[n, K]^T      (both operands K-contiguous, K a multiple of 64)
//
// At these sizes the machine is short of tiles, not of matrix cores: 128 x 320 tiles -- right for T = 2048, one per CU --
// are 128 workgroups at 1000 rows and 16 at 100, and a launch takes 50 us however few there are. So the tile comes in
// sizes from 64 x 32 to 128 x 256, and the host takes the one whose grid fills the 256 CUs in the fewest, cheapest rounds
// (tile_gemm_pick below). What bounds a tile is the bytes its CU pulls in, (BM + BN) x K x 2: a CU has about 64 KB of loads in
// flight whatever the LDS would hold, and a line that no CU of the XCD has asked for yet is about a microsecond away -- 60
// GB/s, where lines that are in the L2 arrive at 100 (measured with the MFMAs and the LDS reads taken out: 0.58 us per
// slice of a 128 x 160 tile, 0.37 with the weight L2-resident; the MFMAs alone 0.34).
//
// Eight wavefronts, 16 TB x 16 RB outputs each on v_mfma_f32_16x16x32_bf16 with the weight on M, WM x WN of them over the
// tile and KG over K: two wavefronts per SIMD, and few enough LDS reads per MFMA. K slices of 64 (one 128-byte line per
// row) pass a ring of S stages filled by global_load_lds_dwordx4, 16-byte chunks XOR-swizzled by row; one hand-spelled
// s_waitcnt + s_barrier per stage, the loads that refill the stage just freed and the next step's fragment reads pinned
// between the current step's MFMAs (sched_group_barrier).
//
// Code that runs once per workgroup is kept small: a cold instruction costs about as much as a cold line of data (8 KB of
// straight-line code ~1 us), and with everything unrolled and the wrap-around's 64-bit divisions inlined per row this
// kernel was 56 KB and had 15 us of prologue and epilogue. It is 9-15 KB now and has 5.7 (64 x 64) to 9 us (128 x 160).
//
// QKV: weight rows are dealt to tile rows so that a lane's four sums are [lo(p), lo(p + 1), hi(p), hi(p + 1)] of two adjacent
// rotation pairs (d, d + 32) -- sixteen-column block B of the output is pairs 8 (B % 4) .. + 8 of head B / 4 -- and any
// multiple of sixteen columns will do as a tile.
//
// [rows, 2880] x [2880, 5120] + bias + rotary, us (before: the many-row decode kernel up to 448 rows, 128 x 320 tiles above):
//   128 rows 16.5 (17.5)   192 16.7 (22.1)   256 18.6 (26.6)   333 21.4 (32.3)   512 25.0 (54.0)   777 31.3 (50.9)
//   999 36.9 (49.1)   1100 38.8 (55.0)   1400 43.7 (57.1)   1536 47.4 (57)
// [rows, 4096] x [4096, 2880] + bias (before: the library's GEMM):
//   97 rows 13.8 (15.5)   192 16.5 (32.2)   333 19.0 (29.9)   512 20.5 (25.1)   999 29.8 (35.4)   2048 49.3 (49.7)
#include "out_common.h"
#include "qkv_prefill.h"

namespace tllm {

namespace tile_gemm {
constexpr int BK = 64, LROW = 128;         // K slice; bytes of an LDS row (one slice of one row)
constexpr int CSROW = 34;                  // float2 per row of the cos / sin table (32 frequencies + padding)

// A tile: wavefronts of 16 TB rows x 16 RB columns, WM x WN of them over the tile, KG over K (WM WN KG = 8).
template <int TB_, int RB_, int WM_, int WN_, int KG_>
struct Tile {
  static constexpr int TB = TB_, RB = RB_, WM = WM_, WN = WN_, KG = KG_, NW = 8;
  static_assert(WM * WN * KG == NW && (KG == 2 || KG == 4), "eight wavefronts");
  static constexpr int BM = 16 * TB * WM, BN = 16 * RB * WN;
  static constexpr int KS = KG == 4 ? 2 : 1;                // slices per stage: a wavefront has one k32 step of it
  static constexpr int SLICE = (BM + BN) * LROW, WSLICE = BN * LROW, STAGE = KS * SLICE;
  static constexpr int CS = BM * CSROW * 8, TAIL = BN * 4;  // cos / sin table (in the idle ring, behind the sums); behind the ring: bias
  static constexpr int S_FIT = (160 * 1024 - TAIL) / STAGE, S = S_FIT > 7 ? 7 : S_FIT;
  static constexpr int SMEM = S * STAGE + TAIL;
  // rows of each operand a wavefront loads per stage (of one slice), eight to an instruction, the last one may be half
  static constexpr int XR = BM * KS / NW, WR = BN * KS / NW, LX = (XR + 7) / 8, LW = (WR + 7) / 8, LPW = LX + LW;
  static_assert(XR % 4 == 0 && WR % 4 == 0 && S >= 3 && (S - 1) * LPW < 64, "three stages resident, and their loads countable");
  // the epilogue passes the sums through the ring, BP of a wavefront's row blocks at a time
  static constexpr int per_block = NW * RB * 1024, BP_FIT = (S * STAGE - CS) / per_block, BP = BP_FIT >= TB ? TB : BP_FIT >= TB / 2 ? TB / 2 : TB / 4, PASSES = TB / BP;
  static_assert(BP >= 1 && BP * per_block + CS <= S * STAGE && PASSES * BP == TB, "sums of a pass fit the ring");
};
}  // namespace tile_gemm

enum : int { kGemmLinear = 0, kGemmYarn = 1, kGemmTable = 2, kGemmResidual = 3 };   // plain | QKV, cos / sin from YaRN parameters | ... from tables | plain + residual (a.k, row stride a.k_rs)

template <int N, int LPW>
__device__ __forceinline__ void wait_slices_left(int left) {     // at most `left` (<= N) slices of LPW loads still in flight
  if constexpr (N == 0) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  } else {
    if (left >= N) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N * LPW) : "memory");
    else wait_slices_left<N - 1, LPW>(left);
  }
}

// TURN: the row tiles begin their walks over K at different places (tile_gemm_spread).
template <class C, int MODE, bool TURN>
__global__ __launch_bounds__(512) void tile_gemm_kernel(QkvArgs a, RopeArgs ra, YarnFreqs fr, int tiles_m, int tiles_n, int group, int n_blocks) {
  using namespace tile_gemm;
  constexpr bool QKV = MODE == kGemmYarn || MODE == kGemmTable;
  constexpr int TB = C::TB, RB = C::RB, KG = C::KG, KS = C::KS, BM = C::BM, BN = C::BN, S = C::S, STAGE = C::STAGE, SLICE = C::SLICE, WSLICE = C::WSLICE;
  constexpr int LX = C::LX, LPW = C::LPW, NB = BN / 16;
  constexpr int NMF = TB * RB, NRD = TB + RB;               // MFMAs and fragment reads per k32 step
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave % KG, wn = wave / KG % C::WN, wm = wave / (KG * C::WN);
  const int m16 = lane & 15, g = lane >> 4;

  // Consecutive block ids go to the eight XCDs in turn: give each XCD a contiguous run of tiles, row tiles fastest, so
  // that the tiles that read the same weight columns share an L2 and the weight leaves HBM once. Of many row tiles `group` at a
  // time, so that an XCD's tiles -- about a rectangle then -- share the rows as well (tile_gemm_group).
  const int tiles = gridDim.x, xcd = blockIdx.x & 7, per = tiles >> 3, extra = tiles & 7;
  const int id = xcd * per + (xcd < extra ? xcd : extra) + (blockIdx.x >> 3);
  // (The second division only where there are groups: it is on the first loads' way, 97 rows of [4096, 2880] 13.7 us without it, 14.0 with.)
  int first_m = 0, group_m = tiles_m, in_group = id;
  if (group < tiles_m) {
    const int grp = id / (group * tiles_n);
    first_m = grp * group;
    in_group -= first_m * tiles_n;
    group_m = tiles_m - first_m < group ? tiles_m - first_m : group;
  }
  const int tile_n = in_group / group_m, tile_m = first_m + in_group % group_m;
  const int64_t row0 = static_cast<int64_t>(tile_m) * BM;
  const int block0 = tile_n * NB;
  const int n_slices = a.hidden / BK, n_iter = (n_slices + KS - 1) / KS;
  const unsigned pitch = static_cast<unsigned>(a.hidden) * 2;

  // Where in K the walk begins, in stages
  const int rot = TURN ? tile_m * n_iter / tiles_m : 0;

  // weight row of tile row i (a block past the last one repeats it; its columns are never stored)
  auto weight_row = [&](int i) {
    int B = block0 + (i >> 4);
    if (B >= n_blocks) B = n_blocks - 1;
    const int i16 = i & 15;
    if constexpr (!QKV) return 16 * B + i16;
    else return (B >> 2) * 64 + 8 * (B & 3) + 2 * (i16 >> 2) + (i16 & 1) + 32 * ((i16 >> 1) & 1);
  };

  // ---- loads. Instruction j of a wavefront fills 1 KB of a slice: eight rows, lane L at row L / 8 of them, chunk position
  // L % 8, where chunk (L % 8) ^ swz(row) belongs. Two slices to a stage: wavefronts 0-3 load the first, 4-7 the second.
  constexpr int XR = C::XR, WR = C::WR;
  const int lw = KS == 2 ? wave & 3 : wave, ls = KS == 2 ? wave >> 2 : 0;
  const unsigned char* const x_base = reinterpret_cast<const unsigned char*>(a.x) + row0 * a.hidden * 2;
  const unsigned char* const w_base = reinterpret_cast<const unsigned char*>(a.W);
  unsigned soff[LPW];
#pragma unroll
  for (int j = 0; j < LPW; ++j) {
    const bool is_x = j < LX;
    const int r = (is_x ? lw * XR + 8 * j : lw * WR + 8 * (j - LX)) + (lane >> 3);
    const unsigned c = static_cast<unsigned>((lane & 7) ^ swz(r)) * 16u;
    if (is_x) {
      int64_t lr = r;
      if (row0 + lr >= a.rows) lr = a.rows - 1 - row0;      // valid memory; these result rows are never stored
      soff[j] = static_cast<unsigned>(lr) * pitch + c;
    } else {
      soff[j] = static_cast<unsigned>(weight_row(r)) * pitch + c;
    }
  }
  // The walk's stage number `st`, which is stage `at` of K, goes into ring place `place`. Nothing is requested behind the last one:
  // the test sits inside the assembly so that the schedule around the load stays one basic block.
  auto issue_load = [&](int st, int at, int place, int j) {
    const bool is_x = j < LX;
    int slice = KS * at + ls;
    if (KS == 2 && slice >= n_slices) slice = n_slices - 1; // an odd number of slices: the last stage's second one is not used
    const unsigned dst = static_cast<unsigned>(reinterpret_cast<uintptr_t>(smem)) + place * STAGE + ls * SLICE +
                         (is_x ? WSLICE + (lw * XR + 8 * j) * LROW : (lw * WR + 8 * (j - LX)) * LROW);
    const unsigned char* sb = (is_x ? x_base : w_base) + static_cast<int64_t>(slice) * (BK * 2);
    const bool half = is_x ? 8 * j + 8 > XR : 8 * (j - LX) + 8 > WR;
    if (half)                                               // known at compile time; every lane is active here, before and after
      asm volatile("s_cmp_lt_i32 %3, %4\n\ts_cbranch_scc0 .Lskip%=\n\ts_mov_b32 m0, %0\n\ts_mov_b32 exec_hi, 0\n\t"
                   "global_load_lds_dwordx4 %1, %2\n\ts_mov_b32 exec_hi, -1\n.Lskip%=:" ::"s"(dst), "v"(soff[j]), "s"(sb), "s"(st), "s"(n_iter)
                   : "memory", "m0", "scc");
    else
      asm volatile("s_cmp_lt_i32 %3, %4\n\ts_cbranch_scc0 .Lskip%=\n\ts_mov_b32 m0, %0\n\ts_nop 0\n\t"
                   "global_load_lds_dwordx4 %1, %2\n.Lskip%=:" ::"s"(dst), "v"(soff[j]), "s"(sb), "s"(st), "s"(n_iter)
                   : "memory", "m0", "scc");
  };

  f32x4 acc[RB][TB];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb)
#pragma unroll
    for (int tb = 0; tb < TB; ++tb) acc[rb][tb] = f32x4{0.f, 0.f, 0.f, 0.f};

  // Fragment addressing: lane group g supplies chunk 4 kk + (g >> 1 | (g & 1) << 1) of a slice's row, which keeps the
  // sixteen lanes a 128-bit LDS read is served by (0-7 with 32-39, ...) on different banks under the row swizzle.
  const int gc = (g >> 1) | ((g & 1) << 1);
  int fx_o[TB], fw_o[RB];
#pragma unroll
  for (int tb = 0; tb < TB; ++tb) {
    const int r = 16 * (TB * wm + tb) + m16;
    fx_o[tb] = WSLICE + r * LROW + ((gc ^ swz(r)) << 4);
  }
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) {
    const int r = 16 * (RB * wn + rb) + m16;
    fw_o[rb] = r * LROW + ((gc ^ swz(r)) << 4);
  }
  bf16x8 fx[2][TB], fw[2][RB];
  auto read_frag = [&](int buf, const unsigned char* st, int kk, int i) {
    if (i < TB) fx[buf][i < TB ? i : 0] = *reinterpret_cast<const bf16x8*>(st + (fx_o[i < TB ? i : 0] ^ (kk << 6)));
    else fw[buf][i < TB ? 0 : i - TB] = *reinterpret_cast<const bf16x8*>(st + (fw_o[i < TB ? 0 : i - TB] ^ (kk << 6)));
  };
  // One k32 step on the fragments in buffer `cur`. Behind its first MFMAs go the reads of the next step's fragments (k32
  // step nkk of the slice at nsl); loads [l0, l1) of the stage handed on spread over all of them.
  auto step = [&](auto cur_c, const unsigned char* nsl, int nkk, auto l0_c, auto l1_c, int stage_it, int stage_at, int stage) {
    constexpr int cur = decltype(cur_c)::value, l0 = decltype(l0_c)::value, l1 = decltype(l1_c)::value;
    constexpr int RPM = (NRD + NMF - 1) / NMF > 1 ? (NRD + NMF - 1) / NMF : 1;   // fragment reads behind an MFMA
#pragma unroll
    for (int m = 0; m < NMF; ++m) {
      const int rb = m / TB, tb = m % TB;
      acc[rb][tb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[cur][rb], fx[cur][tb], acc[rb][tb], 0, 0, 0);
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);             // one MFMA
#pragma unroll
      for (int i = 0; i < NRD; ++i) {
        if (i / RPM != m) continue;
        read_frag(cur ^ 1, nsl, nkk, i);
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);           // an LDS read
      }
#pragma unroll
      for (int i = l0; i < l1; ++i) {
        if ((i - l0) * NMF / (l1 - l0) != m) continue;
        issue_load(stage_it, stage_at, stage, i);
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);           // a VMEM read
      }
    }
  };
  using std::integral_constant;

  // ---- prologue. Nothing here may wait for a vector load before the first slice has to: a wait counts back from the
  // youngest load. The bias value goes out first and is not looked at until the epilogue; the rows' positions come through
  // the scalar cache; then the slices; then the cos / sin arithmetic in their shadow.
  bf16 bias_raw;
  {
    const bf16* bp = a.bias ? a.bias : a.W;                          // absent: a valid address instead of a branch
    bias_raw = bp[weight_row(tid < BN ? tid : BN - 1)];
  }
  // ... as does the residual of the thread's first sixteen outputs, where the registers allow it (the epilogue's row and block of i = tid)
  constexpr bool RES = MODE == kGemmResidual, RES_EARLY = RES && BM == 64;
  const bool res_vec = RES && reinterpret_cast<uintptr_t>(a.k) % 16 == 0 && a.k_rs % 8 == 0;
  bf16x8 res_early[2];
  if constexpr (RES_EARLY) {
    const int b = (tid >> 4) % NB, tbw = (tid >> 4) / NB, r = 16 * (TB * (tbw / C::BP) + tbw % C::BP) + (tid & 15);
    const int64_t grow = row0 + r < a.rows ? row0 + r : a.rows - 1;
    const int B = block0 + b < n_blocks ? block0 + b : n_blocks - 1;
    const bf16* const from = res_vec ? a.k + grow * a.k_rs + 16 * B : a.x;       // (else looked at element by element, later)
    res_early[0] = *reinterpret_cast<const bf16x8*>(from);
    res_early[1] = *reinterpret_cast<const bf16x8*>(from + 8);
  }
  const int first = n_iter < S ? n_iter : S;
  int ahead = rot;                                                  // the stage of K that is loaded next
  auto turn = [&](int next) { ahead = TURN ? (ahead + 1 == n_iter ? 0 : ahead + 1) : next; };
#pragma unroll 1
  for (int s = 0; s < first; ++s) {
#pragma unroll
    for (int j = 0; j < LPW; ++j) issue_load(s, ahead, s, j);
    turn(s + 1);
  }
  // cos / sin of (row, frequency), computed while the first slices arrive and kept in registers. Wavefront w: rows BM / 8 w
  // .. of the tile; lane: frequency lane % 32, rows 2 j + lane / 32 of those. The rows' positions come through the scalar
  // cache and are used as they are when all of them lie in [0, max_ctx), which one comparison of their unsigned maximum
  // says; otherwise (wrap-around) the epilogue fills the table in a rolled loop: the 64-bit divisions inlined here would be 30 KB
  // of code to fetch, executed or not.
  constexpr int RPW = BM / 8, CSN = RPW / 2;                // rows of a wavefront: 8 or 16
  static_assert(RPW == 8 || RPW == 16, "one batch of scalar loads");
  const int64_t first_row = row0 + RPW * wave;
  const int f = lane & 31;
  float2 csr[CSN];
  bool plain = true;
  if (QKV && a.has_rope) {
    int pos[RPW];
    plain = rope_positions_uniform<RPW>(ra, first_row, a.rows, pos);
#pragma unroll
    for (int j = 0; j < CSN; ++j) csr[j] = rope_cos_sin_at<MODE == kGemmTable>(ra, fr, plain ? (lane < 32 ? pos[2 * j] : pos[2 * j + 1]) : 0, f);
  }
  wait_slices_left<S - 1, LPW>(first - 1);
  asm volatile("s_barrier" ::: "memory");
  // Where this wavefront's k32 step is in a stage
  auto slice_at = [&](int stage) { return smem + stage * STAGE + (KG == 4 ? (kg >> 1) * SLICE : 0); };
  const int kk0 = kg & 1;
#pragma unroll
  for (int i = 0; i < NRD; ++i) read_frag(0, slice_at(0), kk0, i);

  // ---- steady state. Ahead of a step -- whose reads are the next stage's fragments -- the stage's one barrier: this
  // wavefront's share of the next stage has landed and its reads of this one are done, then everyone's. The stage vacated
  // is refilled behind it.
  typedef integral_constant<int, 0> I0;
  typedef integral_constant<int, 1> I1;
  typedef integral_constant<int, LPW> IL;
  auto stage_barrier = [&](int it) {                                 // ... with at most min(S - 2, stages behind it + 1) in flight
    const int left = n_iter - 2 - it;
    wait_slices_left<S - 2, LPW>(left > 0 ? left : 0);
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  auto next = [](int c) { return c + 1 == S ? 0 : c + 1; };
  int c = 0;
  // KG == 4, an odd number of slices: the last stage of K has no second one. Half of the wavefronts sit it out, or, where it is met in
  // the middle of the walk, multiply zeros.
  const bool lacks = KG == 4 && n_slices % 2 && kg >= 2;
  const int live = !TURN && lacks ? n_iter - 1 : n_iter, none_at = TURN && lacks ? n_iter - 1 - rot : -1;
  auto no_second_slice = [&](auto buf_c) {
    constexpr int buf = decltype(buf_c)::value;
    const bf16x8 zero = {};
#pragma unroll
    for (int i = 0; i < TB; ++i) fx[buf][i] = zero;
#pragma unroll
    for (int i = 0; i < RB; ++i) fw[buf][i] = zero;
  };
  for (int it = 0; it < n_iter; it += 2) {                           // the fragment buffers alternate, so stages go in pairs
    int n = next(c);
    stage_barrier(it);
    if (TURN && it == none_at) no_second_slice(I0{});
    if (it < live) step(I0{}, slice_at(n), kk0, I0{}, IL{}, it + S, TURN ? ahead : it + S, c);   // (behind the last stage its reads are not used)
    turn(it + S + 1);
    c = n;
    n = next(c);
    stage_barrier(it + 1);
    if (TURN && it + 1 == none_at) no_second_slice(I1{});
    if (it + 1 < live) step(I1{}, slice_at(n), kk0, I0{}, IL{}, it + 1 + S, TURN ? ahead : it + 1 + S, c);
    turn(it + S + 2);
    c = n;
  }
  float* const bias_s = reinterpret_cast<float*>(smem + S * STAGE);
  if (tid < BN) bias_s[tid] = a.bias ? static_cast<float>(bias_raw) : 0.f;

  // ---- epilogue, BP row blocks of every wavefront at a time: the sums go to LDS as they are, and a rolled loop over (row,
  // sixteen-column block) adds the KG shares in a fixed order, adds the bias, rotates, rounds once and stores 2 x 16 bytes.
  const int64_t slot_off = !QKV ? 0 : qkv_slot(a, ra) * a.kv_slot_stride;
  const bool vec_ok = (reinterpret_cast<uintptr_t>(a.q) % 16 == 0) && a.q_rs % 8 == 0 &&
                      (!QKV || ((reinterpret_cast<uintptr_t>(a.k) % 16 == 0) && (reinterpret_cast<uintptr_t>(a.v) % 16 == 0) &&
                                               a.k_rs % 8 == 0 && a.v_rs % 8 == 0 && a.kv_slot_stride % 8 == 0));
  f32x4* const sums = reinterpret_cast<f32x4*>(smem);
  constexpr int BP = C::BP;
  float2* const cs_tab = reinterpret_cast<float2*>(smem + BP * C::per_block);
#pragma unroll
  for (int pass = 0; pass < C::PASSES; ++pass) {
    __syncthreads();                                                 // the ring, or the pass before, is done with
    if (QKV && a.has_rope && pass == 0) {
      float2* const mine = cs_tab + (RPW * wave + (lane >> 5)) * CSROW + f;
      if (plain) {
#pragma unroll
        for (int j = 0; j < CSN; ++j) mine[2 * j * CSROW] = csr[j];
      } else {
#pragma unroll 1
        for (int j = 0; j < CSN; ++j) {
          int64_t gi = first_row + 2 * j + (lane >> 5);
          if (gi >= a.rows) gi = a.rows - 1;
          float cv, sv;
          rope_cos_sin(ra, fr, rope_position(ra, gi), f, &cv, &sv);
          mine[2 * j * CSROW] = make_float2(cv, sv);
        }
      }
    }
    // place of (wavefront column, row half, block, K share): its 64 lanes' sums in a row
#pragma unroll
    for (int rb = 0; rb < RB; ++rb)
#pragma unroll
      for (int tb = 0; tb < BP; ++tb) sums[((((wm * BP + tb) * NB + wn * RB + rb) * KG) + kg) * 64 + lane] = acc[rb][BP * pass + tb];
    __syncthreads();
#pragma unroll 1
    for (int i = tid; i < C::WM * BP * 16 * NB; i += 512) {
      const int r16 = i & 15, b = (i >> 4) % NB, tbw = (i >> 4) / NB;  // row of the block, column block, row block
      const int r = 16 * (TB * (tbw / BP) + BP * pass + tbw % BP) + r16;
      const int B = block0 + b;
      const int64_t grow = row0 + r;
      if (B >= n_blocks || grow >= a.rows) continue;
      const f32x4* from = sums + (tbw * NB + b) * KG * 64 + r16;
      float v[16];
#pragma unroll
      for (int q = 0; q < 4; ++q) {                                  // four columns each
        f32x4 t = from[16 * q];
#pragma unroll
        for (int k = 1; k < KG; ++k) t += from[64 * k + 16 * q];
        t += *reinterpret_cast<const f32x4*>(bias_s + 16 * b + 4 * q);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[4 * q + e] = t[e];
      }
      bf16x8 o0, o1;                                                 // QKV: eight low dims and their partners 32 up; plain: columns 0-7, 8-15
      bf16 *d0, *d1;
      if constexpr (RES) {
        const bf16* const from = a.k + grow * a.k_rs + 16 * B;
        bf16x8 r0, r1;
        if (RES_EARLY && res_vec && pass == 0 && i == tid) {
          r0 = res_early[0];
          r1 = res_early[1];
        } else if (res_vec) {
          r0 = *reinterpret_cast<const bf16x8*>(from);
          r1 = *reinterpret_cast<const bf16x8*>(from + 8);
        } else {
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            r0[e] = from[e];
            r1[e] = from[8 + e];
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          v[e] += static_cast<float>(r0[e]);
          v[8 + e] += static_cast<float>(r1[e]);
        }
      }
      if constexpr (!QKV) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          o0[e] = static_cast<bf16>(v[e]);
          o1[e] = static_cast<bf16>(v[8 + e]);
        }
        d0 = a.q + grow * a.q_rs + 16 * B;
        d1 = d0 + 8;
      } else {
        const int head = B >> 2, dim = 8 * (B & 3);
        if (a.has_rope && head < a.n_q_heads + a.n_kv_heads) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const f32x4 cs = *reinterpret_cast<const f32x4*>(cs_tab + r * CSROW + dim + 2 * q);   // cos, sin of two frequencies
            const float l0 = v[4 * q], l1 = v[4 * q + 1], h0 = v[4 * q + 2], h1 = v[4 * q + 3];
            v[4 * q] = l0 * cs[0] - h0 * cs[1];
            v[4 * q + 1] = l1 * cs[2] - h1 * cs[3];
            v[4 * q + 2] = h0 * cs[0] + l0 * cs[1];
            v[4 * q + 3] = h1 * cs[2] + l1 * cs[3];
          }
        }
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          o0[e] = static_cast<bf16>(v[4 * (e >> 1) + (e & 1)]);
          o1[e] = static_cast<bf16>(v[4 * (e >> 1) + (e & 1) + 2]);
        }
        if (head < a.n_q_heads) d0 = a.q + grow * a.q_rs + static_cast<int64_t>(head) * 64 + dim;
        else if (head < a.n_q_heads + a.n_kv_heads) d0 = a.k + grow * a.k_rs + slot_off + static_cast<int64_t>(head - a.n_q_heads) * 64 + dim;
        else d0 = a.v + grow * a.v_rs + slot_off + static_cast<int64_t>(head - a.n_q_heads - a.n_kv_heads) * 64 + dim;
        d1 = d0 + 32;
      }
      if (vec_ok) {
        *reinterpret_cast<bf16x8*>(d0) = o0;
        *reinterpret_cast<bf16x8*>(d1) = o1;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          d0[e] = o0[e];
          d1[e] = o1[e];
        }
      }
    }
  }
}

namespace {
// Row tiles that a column of tiles takes before the next column begins. All of them, up to 16: the rows that an XCD's 32 tiles of a round
// read are then few enough. Beyond, eight; us, all and eight, 17 - 50 row tiles: [rows, 2880] x [2880, 5120] 2300 rows 81.4 / 76.9, 2800 90.5 /
// 86.3, 4300 142.9 / 132.6, 6300 190.6 / 180.5; 2880 x 1024 1411 rows 16.7 / 15.1, 2500 24.5 / 20.6; 4096 x 5120 2300 99.6 / 91.2 (six and four
// the same within 1 %; with fewer row tiles 4096 x 2880 1100 rows 36.4 / 37.8, 2048 50.9 / 50.3). An operand that is small anyway has
// nothing to gain before the rows are many: 1024 x 1024 1411 rows 8.2 / 8.3, 2300 11.3 / 10.8.
int64_t tile_gemm_group(int64_t tiles_m, int64_t weight) { return tiles_m > (weight > 2000000 ? 16 : 32) ? 8 : tiles_m; }

template <class C, int MODE, bool TURN>
int launch_one(const char* what, const QkvArgs& a, const RopeArgs& ra, const YarnFreqs& fr, int n_blocks, hipStream_t st) {
  static std::atomic<uint64_t> done{0};
  const hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(tile_gemm_kernel<C, MODE, TURN>), C::SMEM, done);
  TLLM_REQUIRE(e == hipSuccess, TLLM_E_LAUNCH, "%s: cannot raise LDS limit: %s", what, hipGetErrorString(e));
  const int64_t tiles_m = (a.rows + C::BM - 1) / C::BM, tiles_n = (n_blocks * 16 + C::BN - 1) / C::BN;
  const int64_t group = tile_gemm_group(tiles_m, static_cast<int64_t>(n_blocks) * 16 * a.hidden);
  TLLM_REQUIRE(tiles_m * tiles_n < (1ll << 31), TLLM_E_SHAPE, "%s: too many tiles", what);
  hipLaunchKernelGGL((tile_gemm_kernel<C, MODE, TURN>), dim3((unsigned)(tiles_m * tiles_n)), dim3(512), C::SMEM, st, a, ra, fr, (int)tiles_m, (int)tiles_n, (int)group, n_blocks);
  return check_launch(what);
}

// Which tile. A tile's time is what its CU pulls through its L2 port -- (BM + BN) rows of K -- at the 60 GB/s that cold lines
// arrive with (2.15 ns per row and slice of 64 K, the same within 5 % from 64 x 32 to 128 x 160), plus launch, first
// slice and epilogue, which grow with the tile (5.3 us at 64 x 32, 9 at 128 x 160); a CU holds one tile at a time. Measured on
// [rows, 2880] x [2880, 5120], us, chosen tile against the neighbouring ones:
//   97 rows   64 x 48 15.7   64 x 64 16.9   64 x 32 23.8        256 rows  64 x 80 18.6    64 x 64 28.6    64 x 128 21.5
//   333 rows  64 x 128 21.4  64 x 160 23.5  64 x 96 32.1        512 rows  64 x 160 24.8   128 x 128 27.6  64 x 128 37.8
//   777 rows  128 x 160 31.3 128 x 192 34.3 64 x 160 43.4       999 rows  128 x 160 37.4  128 x 192 39.1  128 x 128 60.7
// (It knows neither walks that are spread over K, 8 % less in the mean, nor groups of row tiles; both came after it was fitted.)
constexpr TileSize kTiles[] = {{64, 32}, {64, 48}, {64, 64}, {64, 80}, {64, 96}, {64, 128}, {64, 160}, {64, 192}, {128, 96}, {128, 128}, {128, 160}, {128, 192}, {128, 224}, {128, 256}};

int64_t tile_ns(int64_t rows, int64_t cols, int64_t k, TileSize t) {
  const int64_t tiles = ((rows + t.bm - 1) / t.bm) * ((cols + t.bn - 1) / t.bn), rounds = (tiles + 255) / 256;
  return 1600 + rounds * (1700 + 20 * (t.bm + t.bn) + (k / 64) * (t.bm + t.bn) * 215 / 100);
}

}  // namespace

TileSize tile_gemm_pick(int64_t rows, int64_t cols, int64_t k, int64_t* ns) {
  TileSize best = kTiles[0];
  *ns = tile_ns(rows, cols, k, best);
  for (const TileSize& t : kTiles) {
    const int64_t c = tile_ns(rows, cols, k, t);
    if (c < *ns) {
      *ns = c;
      best = t;
    }
  }
  return best;
}

namespace {
// Whether the row tiles of a launch begin their walks over K at places spread over it (tile m of M at m / M). In step, the
// workgroups that share weight columns all wait for the same lines from memory; spread, each finds most of K in its XCD's L2, where
// another one has been. It pays while an XCD's share of the weight stays in its 4 MB (16 M elements; below 8 M, with rows 4 or 8 KB
// apart below 10 M, in step was as fast with the weights measured first). 700 MB of weights in turn, so that each comes from memory, in
// step / spread, us: [rows, 4096] x [4096, 2880] 128 rows 16.4 / 15.4, 256 18.9 / 16.4, 450 22.2 / 20.4, 640 29.8 / 25.3; [rows, 2880] x [2880,
// 5120] 192 17.5 / 15.2, 300 23.1 / 20.0, 640 30.6 / 27.1; 6144 x 2048 640 35.9 / 29.5; and 4096 x 5120 256 rows 24.6 / 29.0, 8192 x 2048 513 34.9 /
// 42.1, 8192 x 1536 300 24.7 / 27.0, 1024 x 8192 256 11.5 / 12.0. A weight that stays in the 256 MB behind the L2 from one call to the
// next has less to gain: 2880 x 2880 256 rows, 200 MB in turn, 11.5 / 12.6, 2048 x 5120 11.3 / 13.0.
// In step, a last row tile that is mostly empty is ahead of the others and fetches for them, so that spreading wants one that is
// filled, the more the fewer row tiles there are and the fewer columns a tile has. In step / spread, mean and worst of 39 weights: two
// row tiles, 113 rows (49 in the last) 1.018, 0.98; three, 160 (32) of 48 columns 1.014, 0.98, 168 (40) of 32 columns 1.007, 0.97; four, 200
// (8) 0.985, 0.91, 220 (28) 1.038, 0.98; five, 257 (1) 1.006, 0.90, 272 (16) 1.045, 0.97; six, 330 (10) 1.058, 0.96; 256 1.14, 640 1.16.
// 128-row tiles up to 128 columns: 5 tiles of 2880 x 5120 640 rows 30.6 / 27.1, six of them (720) 29.8 / 29.4, 2880 x 4096 720 rows 28.5 /
// 26.0; 4096 x 2880 1300 rows (20 in the last) 35.7 / 38.8.
// The order in which a row's products are summed then depends on its row tile: equal rows of one call agree to rounding, not to the bit.
bool tile_gemm_spread(int64_t rows, int64_t cols, int64_t k, TileSize t) {
  const int64_t last = (rows - 1) % t.bm + 1, tiles_m = (rows + t.bm - 1) / t.bm, weight = cols * k;
  if (tiles_m < 2 || weight < 8000000 || weight > 16000000 || (weight < 10000000 && k % 2048 == 0) || k > 6144) return false;
  if (t.bm == 64) {
    if (tiles_m <= 3) return last >= (tiles_m == 2 ? 48 : t.bn == 32 ? 40 : t.bn == 48 ? 32 : 24);
    return k >= 1536 && last >= (tiles_m == 4 ? 28 : tiles_m == 5 ? 16 : tiles_m == 6 ? 8 : 1);
  }
  return t.bn <= 128 && last >= 80 && (tiles_m <= 5 || weight <= 12000000);
}

template <int MODE>
int launch_mode(const char* what, const QkvArgs& a, const RopeArgs& ra, const YarnFreqs& fr, int n_blocks, hipStream_t st) {
  int64_t ns;
  TileSize t = tile_gemm_pick(a.rows, static_cast<int64_t>(n_blocks) * 16, a.hidden, &ns);
  const bool spread = tile_gemm_spread(a.rows, static_cast<int64_t>(n_blocks) * 16, a.hidden, t);
#define TLLM_TILE(...)                                                                                                  \
  if (typedef tile_gemm::Tile<__VA_ARGS__> C; t.bm == C::BM && t.bn == C::BN) {                          \
    constexpr bool CAN = C::BM == 64 || C::BN <= 128;   /* (one kernel for both costs 1 - 4 % in step) */          \
    return CAN && spread ? launch_one<C, MODE, CAN>(what, a, ra, fr, n_blocks, st) : launch_one<C, MODE, false>(what, a, ra, fr, n_blocks, st); \
  }
  TLLM_TILE(2, 2, 2, 1, 4)
  TLLM_TILE(2, 3, 2, 1, 4)
  TLLM_TILE(4, 2, 1, 2, 4)
  TLLM_TILE(2, 5, 2, 1, 4)
  TLLM_TILE(4, 3, 1, 2, 4)
  TLLM_TILE(2, 4, 2, 2, 2)
  TLLM_TILE(2, 5, 2, 2, 2)
  TLLM_TILE(2, 6, 2, 2, 2)
  TLLM_TILE(4, 3, 2, 2, 2)
  TLLM_TILE(4, 4, 2, 2, 2)
  TLLM_TILE(4, 5, 2, 2, 2)
  TLLM_TILE(4, 6, 2, 2, 2)
  TLLM_TILE(4, 7, 2, 2, 2)
  TLLM_TILE(4, 8, 2, 2, 2)
#undef TLLM_TILE
  set_error("%s: no kernel for a tile of %d x %d", what, t.bm, t.bn);
  return TLLM_E_SHAPE;
}
}  // namespace

int64_t tile_gemm_ns(int64_t rows, int64_t cols, int64_t k) {
  int64_t ns;
  tile_gemm_pick(rows, cols, k, &ns);
  return ns;
}

int launch_tile_gemm_qkv(const char* what, const QkvArgs& a, const RopeArgs& ra, const YarnFreqs& fr, hipStream_t st) {
  const int n_blocks = (a.n_q_heads + 2 * a.n_kv_heads) * 4;
  return a.has_rope && !ra.use_yarn ? launch_mode<kGemmTable>(what, a, ra, fr, n_blocks, st) : launch_mode<kGemmYarn>(what, a, ra, fr, n_blocks, st);
}

}  // namespace tllm

using namespace tllm;

extern "C" int tllm_qkv_gemm_tile(int prefill, int64_t rows, int64_t hidden, int n_q_heads, int n_kv_heads, int head_dim) {
  const int heads = n_q_heads + 2 * n_kv_heads;
  if (rows < 1 || hidden < 1 || heads < 1 || !(prefill ? qkv_prefill_tiles : qkv_decode_tiles)(rows, hidden, heads, head_dim)) return 0;
  int64_t ns;
  const TileSize t = tile_gemm_pick(rows, static_cast<int64_t>(heads) * 64, hidden, &ns);
  return t.bm << 16 | t.bn;
}

extern "C" int tllm_linear_gemm_tile(int64_t rows, int64_t in_dim, int64_t out_dim) {
  int64_t ns;
  const TileSize t = tile_gemm_pick(rows, out_dim, in_dim, &ns);
  return t.bm << 16 | t.bn;
}

namespace tllm {
// What tllm_linear_bf16 takes, of K, outputs and alignment.
bool linear_fits_tiles(const void* x, const void* W, int64_t rows, int64_t in_dim, int64_t out_dim) {
  return rows < (1ll << 31) && in_dim >= 64 && in_dim % 64 == 0 && out_dim >= 16 && out_dim % 16 == 0 && in_dim * out_dim * 2 < (1ll << 32) &&
         in_dim * 512 < (1ll << 32) && aligned16(x) && aligned16(W);
}

int launch_tile_gemm_out(const char* what, const OutArgs& o, hipStream_t st) {
  QkvArgs a{};
  a.x = o.x;
  a.W = static_cast<const bf16*>(o.W);
  a.bias = o.bias;
  a.k = const_cast<bf16*>(o.res);
  a.k_rs = o.res_rs;
  a.q = o.out;
  a.q_rs = o.out_rs;
  a.rows = o.rows;
  a.hidden = o.in_dim;
  const int n_blocks = o.out_dim / 16;
  return o.res ? launch_mode<kGemmResidual>(what, a, RopeArgs{}, YarnFreqs{}, n_blocks, st) : launch_mode<kGemmLinear>(what, a, RopeArgs{}, YarnFreqs{}, n_blocks, st);
}
}  // namespace tllm

extern "C" int tllm_gemm_tile_group(int64_t rows, int64_t in_dim, int64_t out_dim) {
  int64_t ns;
  const int64_t bm = tile_gemm_pick(rows, out_dim, in_dim, &ns).bm;
  return static_cast<int>(tile_gemm_group((rows + bm - 1) / bm, out_dim * in_dim));
}

extern "C" int tllm_gemm_tile_spread(int64_t rows, int64_t in_dim, int64_t out_dim) {
  int64_t ns;
  return tile_gemm_spread(rows, out_dim, in_dim, tile_gemm_pick(rows, out_dim, in_dim, &ns));
}

extern "C" int tllm_linear_bf16(const void* x, const void* W, const void* b, void* out, int64_t out_row_stride, int64_t rows, int64_t in_dim,
                                int64_t out_dim, void* stream) {
  TLLM_REQUIRE(rows >= 0 && rows < (1ll << 31) && in_dim >= 64 && in_dim % 64 == 0 && out_dim >= 16 && out_dim % 16 == 0, TLLM_E_SHAPE,
               "linear: rows %lld, in_dim %lld (a multiple of 64), out_dim %lld (of 16)", (long long)rows, (long long)in_dim, (long long)out_dim);
  TLLM_REQUIRE(in_dim * out_dim * 2 < (1ll << 32) && in_dim * 512 < (1ll << 32), TLLM_E_SHAPE, "linear: weight of 4 GiB or more");
  if (rows == 0) return TLLM_OK;
  TLLM_REQUIRE(x && W && out && out_row_stride >= out_dim, TLLM_E_ARG, "linear: x, W, out must not be NULL and out_row_stride not below out_dim");
  TLLM_REQUIRE(aligned16(x) && aligned16(W), TLLM_E_ALIGN, "linear: x and W must be 16-byte aligned");
  QkvArgs a{};
  a.x = static_cast<const bf16*>(x);
  a.W = static_cast<const bf16*>(W);
  a.bias = static_cast<const bf16*>(b);
  a.q = static_cast<bf16*>(out);
  a.q_rs = out_row_stride;
  a.rows = rows;
  a.hidden = static_cast<int>(in_dim);
  return launch_mode<kGemmLinear>("linear", a, RopeArgs{}, YarnFreqs{}, static_cast<int>(out_dim / 16), static_cast<hipStream_t>(stream));
}
