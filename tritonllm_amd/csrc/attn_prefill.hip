// Prefill attention with learned sinks and an optional sliding window: many query positions per batch row against
// the keys written so far (attention, attention_tt.py:167-242; kernel :17-164; definition attention_ref.py:4-42):
//
//   query i of a batch row sits at position p = start_q + i and sees the keys n with
//       n <= p,   n < n_kv_ctx,   n > p - window (when a window is set)
//   s[i, h, n] = sm_scale * <q[i, h], k[n, kv(h)]>                      kv(h) = h / G   (G query heads share a KV head)
//   out[i, h]  = sum_n exp(s - m) v[n, kv(h)] / (sum_n exp(s - m) + exp(sink[h] - m)),    m = max(sink[h], max_n s)
//
// The reference transposes q, k and v into head-major copies, pads them to the block size and runs one program per
// (64 queries, query head). Here the kernel reads q as the QKV projection wrote it ([token, head, 64]) and k / v in
// the cache layout ([token, kv head, 64]), and writes [token, head * 64]: no copies on either side.
//
//   * a workgroup takes 64 (128) consecutive queries of up to four query heads that share a KV head, a wavefront 32 queries
//     of one or two of them; K / V blocks of 64 keys pass through four LDS stages filled by global_load_lds_dwordx4 (no
//     staging registers, no LDS writes; two blocks in flight behind the two being computed, one hand-spelled wait + barrier
//     per two blocks) and serve all heads; the smallest launches share the key blocks of 64 queries x 1 head out to two or
//     four groups of two wavefronts, which meet in LDS at the end (what is bound there is the serial walk over the keys,
//     ~1 us a block);
//   * S^T = K . Q^T on v_mfma_f32_32x32x16_bf16 with the keys on M: a lane then owns ONE query (column) and 16 keys
//     per 32-key block, so the running maximum, the running sum and the rescale factor of the online softmax are
//     lane-local apart from one exchange between the two half-wavefronts;
//   * those accumulator registers are, pairwise, the B operand (P^T) of O^T = V^T . P^T when the MFMA's k slots are read
//     as a permutation of the block's keys, so P never leaves the registers; V stays row-major in LDS and the A operand
//     (V^T: lane = d, 8 keys) comes out of two transposing reads (ds_read_b64_tr_b16: within 16 lanes, lane i receives
//     element i % 4 of the 8 bytes addressed by lanes i / 4, 4 + i / 4, 8 + i / 4, 12 + i / 4);
//   * the running maximum is only raised when a block exceeds it by more than 2^8 (exponents stay far from overflow, the
//     result is the same quotient), so the accumulator is almost never rescaled; the weights are summed, as the bf16
//     values the MFMA multiplies with, two per v_dot2c_f32_bf16 (the long walks' kernel, further down, does both differently);
//   * both tiles are XOR-swizzled in 16-byte chunks: fragment reads are conflict-free (K) or at the two-pass minimum (V);
//   * the KV head is the fastest-varying part of the workgroup index, so with eight KV heads each XCD's L2 holds the
//     K and V of one head; the query tiles with the most keys to visit are launched first.
// start_q is read from device memory (int32 or int64).
#include "common.h"

namespace tllm {

struct AttnPrefillArgs {
  const bf16* q;          // [B, n_q, n_heads, 64]: batch stride q_bs, token stride q_ts (elements), heads adjacent
  const bf16* k;          // [B, n_kv_ctx, n_kv_heads, 64]: batch stride kv_bs, token stride kv_ts
  const bf16* v;
  const bf16* sinks;      // [n_heads] or null (logit 0, attention_tt.py:100-104)
  bf16* out;              // [B, n_q, n_heads * 64]: batch stride out_bs, token stride out_ts
  const void* start_q;    // device scalar
  int start_is_i64;
  int64_t q_bs, q_ts, out_bs, out_ts, kv_bs, kv_ts;
  int batch, n_q, n_kv_ctx, n_kv_heads, group, window;
  float sm_scale;
};

namespace {
constexpr int PBN = 64;               // keys per block
constexpr int KT_BYTES = PBN * 128;   // K tile [key][64 d]
constexpr int VT_BYTES = PBN * 128;   // V tile [key][64 d]
constexpr int PSTAGE = KT_BYTES + VT_BYTES;
constexpr float kLog2e = 1.4426950408889634f;
}  // namespace

constexpr float kRaise = 8.f;         // log2 units by which a block must exceed the running maximum to move it
constexpr float kLift = 7.f;          // where maxima are not taken: how far the reference lies above the maximum it was raised to
constexpr float kNoRef = 3.0e38f;     // no key has been seen: the negated reference (finite, so that a masked logit gives exp2(-inf) and not nan)

// 16-byte chunk swizzle of a V row: a transposing read touches eight consecutive keys x 64 bytes; this spreads them
// over the banks evenly.
__device__ __forceinline__ int v_swizzle(int key) { return (((key >> 1) & 1) << 2) | ((key >> 2) & 3); }

// The value lane l ^ 32 holds: lanes l and l ^ 32 carry the two halves of one query's keys.
__device__ __forceinline__ float other_half(float x, int high) {
  const unsigned u = __builtin_bit_cast(unsigned, x);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);   // r[0]: the low half's x in every lane, r[1]: the high half's
  return __builtin_bit_cast(float, high ? r[0] : r[1]);
}

typedef __attribute__((__vector_size__(4 * sizeof(short)))) short i16x4;
typedef __attribute__((__vector_size__(4 * sizeof(unsigned)))) unsigned u32x4;

// NH: query heads (of one KV head) per wavefront. QG: groups of 32 queries per workgroup, KG: groups that share the key
// blocks out. The NW wavefronts are QG query groups x KG key groups x HS head sets, so a workgroup covers 32 * QG queries of
// NH * HS heads.
template <int NH, int QG, int KG, int NW>
__global__ __launch_bounds__(NW * 64, KG > 2 ? NW / 4 : NW / 2) void attn_prefill_kernel(AttnPrefillArgs a) {
  constexpr int PBM = 32 * QG;                    // queries per workgroup
  constexpr int HS = NW / (QG * KG);              // head sets
  static_assert(HS * QG * KG == NW && (KG == 1 || (NH == 1 && HS == 1)), "wavefronts of a workgroup");
  constexpr int STEP = KG == 1 ? 2 : KG;          // blocks between two barriers
  constexpr int NSTG = 2 * STEP;                  // LDS stages: the step's blocks and the next one's
  constexpr int DPT = KG == 1 ? 16 / NW : 16 * STEP / NW;   // global->LDS load instructions (1 KB each) per wavefront: of every block / of its block of a step
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, h = lane >> 5;

  // workgroup -> (kv head, head sub-group, batch row, query tile); kv head fastest. Long tiles go first; when the whole
  // launch is resident at once (two workgroups per CU), the second workgroup of each CU is taken in the opposite
  // order, so a CU that got a long tile gets a short one next to it.
  const int nsub = a.group / (NH * HS);
  const int ntiles = (a.n_q + PBM - 1) / PBM;
  unsigned id = blockIdx.x;
  const int kvh = id % a.n_kv_heads;
  id /= a.n_kv_heads;
  {
    const unsigned per_round = 256 / (a.n_kv_heads < 256 ? a.n_kv_heads : 256);      // first workgroups of the CUs, per KV head
    const unsigned n = gridDim.x / a.n_kv_heads;
    if (per_round > 0 && n <= 2 * per_round && id >= per_round) id = n + per_round - 1 - id;
  }
  const int sub = id % nsub;
  id /= nsub;
  const int b = id % a.batch;
  id /= a.batch;
  const int tile = ntiles - 1 - static_cast<int>(id);
  const int kgrp = KG == 1 ? 0 : wave / QG;       // the wavefront's key group (KG == 1: wave / QG is its head set)
  const int head0 = kvh * a.group + (KG == 1 ? sub * HS + wave / QG : sub) * NH;

  // ---- Q fragments (B operand: lane = query, 8 d per half-wavefront and k16 step), requested before the start
  // position is read: their addresses do not depend on it, so they travel while that (dependent) load is on its way
  const int q0 = tile * PBM;
  const int qw0 = q0 + (wave % QG) * 32;   // the wavefront's first query
  bf16x8 qf[NH][4];
  {
    int qrow = qw0 + l31;
    qrow = qrow < a.n_q ? qrow : a.n_q - 1;
    const bf16* qp = a.q + b * a.q_bs + static_cast<int64_t>(qrow) * a.q_ts + head0 * 64 + h * 8;
#pragma unroll
    for (int hd = 0; hd < NH; ++hd)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) qf[hd][kk] = *reinterpret_cast<const bf16x8*>(qp + hd * 64 + kk * 16);
  }

  const int start = a.start_is_i64 ? static_cast<int>(*reinterpret_cast<const int64_t*>(a.start_q)) : *reinterpret_cast<const int*>(a.start_q);
  const int p0 = start + qw0;              // the position of the wavefront's first query
  const int q_end = q0 + PBM < a.n_q ? q0 + PBM : a.n_q;
  int kv_hi = start + q_end < a.n_kv_ctx ? start + q_end : a.n_kv_ctx;       // keys the tile's last query sees (exclusive)
  kv_hi = kv_hi > 0 ? kv_hi : 0;
  int kv_lo = a.window > 0 ? start + q0 - a.window + 1 : 0;
  kv_lo = kv_lo > 0 ? kv_lo : 0;
  kv_lo = kv_lo < kv_hi ? kv_lo : kv_hi;
  const int blk_lo = kv_lo / PBN, blk_hi = (kv_hi + PBN - 1) / PBN;
  const int nblk = blk_hi - blk_lo;
  const int key_max = kv_hi - 1;           // rows beyond it are never visible and may hold anything: not loaded

  const bf16* kp = a.k + b * a.kv_bs + kvh * 64;
  const bf16* vp = a.v + b * a.kv_bs + kvh * 64;

  // ---- K / V block movers: global_load_lds_dwordx4 (no staging registers, no LDS writes). One instruction fills
  // 1 KB = 8 tile rows, the lanes' 16 bytes landing at M0 + 16 * lane; the swizzle is applied by choosing which chunk of
  // the row a lane fetches. A stage is the K tile followed by the V tile, so a wavefront's DPT instructions all belong
  // to one of the two.
  const int dma_first = wave * DPT & 15;          // the wavefront's first instruction of the block's sixteen: eight of K, eight of V
  const int dma_block = KG == 1 ? 0 : wave * DPT >> 4;
  const bool dma_v = dma_first >= 8;              // they all belong to one of the two tiles
  const bf16* const dma_src = dma_v ? vp : kp;
  int dma_row[DPT], dma_col[DPT];
  const bf16* dma_ptr[DPT];                       // the lane's chunk of its row of key block 0
#pragma unroll
  for (int j = 0; j < DPT; ++j) {
    const int row = ((dma_first + j) & 7) * 8 + (lane >> 3);
    dma_row[j] = row;
    dma_col[j] = ((lane & 7) ^ (dma_v ? v_swizzle(row) : ((row >> 1) & 7))) * 8;
    dma_ptr[j] = dma_src + static_cast<int64_t>(row) * a.kv_ts + dma_col[j];
  }
  const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(smem)) + dma_first * 1024;
  const int64_t blk_stride = static_cast<int64_t>(PBN) * a.kv_ts;
  auto issue_block = [&](int blk, int stage) {
    const bool whole = blk * PBN + PBN - 1 <= key_max;       // no row of the block lies beyond the last visible key
#pragma unroll
    for (int j = 0; j < DPT; ++j) {
      const bf16* g;
      if (whole) {
        g = dma_ptr[j] + blk * blk_stride;
      } else {
        int key = blk * PBN + dma_row[j];
        key = key < key_max ? key : key_max;
        g = dma_src + static_cast<int64_t>(key) * a.kv_ts + dma_col[j];
      }
      const unsigned m0v = lds0 + stage * PSTAGE + j * 1024;
      asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(m0v), "v"(g) : "memory", "m0");
    }
  };
  // the blocks of the step that starts at block i (counted from blk_lo) into their stages
  auto issue_step = [&](int i) {
    if constexpr (KG == 1) {
#pragma unroll
      for (int j = 0; j < STEP; ++j)
        if (i + j < nblk) issue_block(blk_lo + i + j, (i + j) & (NSTG - 1));
    } else {
      if (i + dma_block < nblk) issue_block(blk_lo + i + dma_block, (i + dma_block) & (NSTG - 1));
    }
  };
  // wait until this wavefront's loads have landed, then meet the others
  auto wait_and_meet = [] { asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); };

  // K fragment (A operand of S^T): lane = key l31 of a 32-key half, 16 bytes at d = kk*16 + h*8
  const int k_row = l31 * 128, k_sw = (l31 >> 1) & 7;
  // V^T fragment (A operand of O^T): lane = d; the transposing read wants from lane j of each 16 the address of
  // four d (quad j % 4 of the lane group's 16) of key j / 4 of the four keys this half-wavefront takes
  const int v_key = 4 * h + ((lane & 15) >> 2);                       // + 16*cc + 8*u + 32*kb
  const int v_d = (l31 & 16) + 4 * (lane & 3);                        // + 32*db

  // ---- running state: lane = query; m in log2 units of the scaled logits
  const float c = a.sm_scale * kLog2e;
  float m_run[NH], l_run[NH];
  f32x16 o[NH][2];
#pragma unroll
  for (int hd = 0; hd < NH; ++hd) {
    m_run[hd] = -INFINITY;
    l_run[hd] = 0.f;
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[hd][db][r] = 0.f;
  }

  issue_step(0);

  {
    // The compiler does not see the direct-to-LDS loads in its count of outstanding loads; were the fragments first
    // used inside the loop, its wait for them there would be "nothing outstanding" and drain the blocks in flight on
    // every step. Pin the wait here, where the first blocks have to land anyway.
#pragma unroll
    for (int hd = 0; hd < NH; ++hd)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) asm volatile("" : "+v"(qf[hd][kk]));
  }

  wait_and_meet();                               // the first step's blocks have landed

  auto process = [&](int blk, int stage) __attribute__((always_inline)) {
    const int key0 = blk * PBN;
    // does any of the wavefront's 32 queries see a key of this block?
    const bool active = key0 <= p0 + 31 && (a.window <= 0 || key0 + PBN - 1 >= p0 - a.window + 1);
    if (active) {
      const unsigned char* ks = smem + stage * PSTAGE;
      const unsigned char* vs = ks + KT_BYTES;
      // S^T[key, query]
      f32x16 s[NH][2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) {
          const bf16x8 kf = *reinterpret_cast<const bf16x8*>(ks + kb * 32 * 128 + k_row + (((kk * 2 + h) ^ k_sw) << 4));
#pragma unroll
          for (int hd = 0; hd < NH; ++hd) {
            if (kk == 0) {
              const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
              s[hd][kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[hd][kk], zero, 0, 0, 0);
            } else {
              s[hd][kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf, qf[hd][kk], s[hd][kb], 0, 0, 0);
            }
          }
        }
      // mask where the block crosses the causal diagonal, the window's trailing edge or the end of the keys
      const bool full = key0 + PBN - 1 <= p0 && key0 + PBN - 1 < a.n_kv_ctx && (a.window <= 0 || key0 >= p0 + 31 - a.window + 1);
      if (!full) {
        const int qp = p0 + l31;
        const int upper = qp < a.n_kv_ctx - 1 ? qp : a.n_kv_ctx - 1;
        const int lower = a.window > 0 ? qp - a.window + 1 : -2147483647;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const int key = key0 + kb * 32 + 8 * (r >> 2) + 4 * h + (r & 3);
            const bool vis = key <= upper && key >= lower;
#pragma unroll
            for (int hd = 0; hd < NH; ++hd) s[hd][kb][r] = vis ? s[hd][kb][r] : -INFINITY;
          }
      }
      // online softmax. First the block maxima of all heads and ONE (rare) branch that raises running maxima; what
      // follows is then a single straight-line region in which the exponentials of one (head, 32-key half) and the
      // P.V MFMAs of the one before it can be issued in turn.
      bool raise[NH];
      float mx[NH];
      bool any = false;
#pragma unroll
      for (int hd = 0; hd < NH; ++hd) {
        float t = -INFINITY;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) t = fmaxf(t, s[hd][kb][r]);
        mx[hd] = fmaxf(t, other_half(t, h)) * c;
        // the maximum moves only when this block tops it by more than kRaise: p stays below 2^kRaise otherwise
        raise[hd] = mx[hd] > m_run[hd] + kRaise;                  // false while mx is -inf (nothing visible yet)
        any = any || raise[hd];
      }
      if (__builtin_amdgcn_ballot_w64(any) != 0) {
#pragma unroll
        for (int hd = 0; hd < NH; ++hd) {
          const float m_new = raise[hd] ? mx[hd] : m_run[hd];
          const float alpha = raise[hd] ? __builtin_amdgcn_exp2f(m_run[hd] - m_new) : 1.f;     // -inf - finite: 0
          m_run[hd] = m_new;
          l_run[hd] *= alpha;
#pragma unroll
          for (int db = 0; db < 2; ++db)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[hd][db][r] *= alpha;
        }
      }
      const bf16x2 one2 = {static_cast<bf16>(1.0f), static_cast<bf16>(1.0f)};
#pragma unroll
      for (int hd = 0; hd < NH; ++hd) {
        const float m_use = m_run[hd] == -INFINITY ? 0.f : m_run[hd];
        float lsum = l_run[hd];
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
          // P^T in bf16 straight into operand registers
          bf16x8 pf[2];
#pragma unroll
          for (int r = 0; r < 16; ++r) pf[r >> 3][r & 7] = static_cast<bf16>(__builtin_amdgcn_exp2f(fmaf(s[hd][kb][r], c, -m_use)));
          // the denominator sums the rounded weights the numerator's MFMA multiplies with, two per instruction
#pragma unroll
          for (int cc = 0; cc < 2; ++cc) {
            lsum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(pf[cc], pf[cc], 0, 1), one2, lsum, false);
            lsum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(pf[cc], pf[cc], 2, 3), one2, lsum, false);
            lsum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(pf[cc], pf[cc], 4, 5), one2, lsum, false);
            lsum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_shufflevector(pf[cc], pf[cc], 6, 7), one2, lsum, false);
          }
          // O^T[d, query] += V^T[d, keys] . P^T[keys, query]
#pragma unroll
          for (int cc = 0; cc < 2; ++cc)
#pragma unroll
            for (int db = 0; db < 2; ++db) {
              i16x4 part[2];
#pragma unroll
              for (int u = 0; u < 2; ++u) {
                const int key = kb * 32 + cc * 16 + u * 8 + v_key;
                const int d = db * 32 + v_d;
                part[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
                    (__attribute__((address_space(3))) i16x4*)(vs + key * 128 + (((d >> 3) ^ v_swizzle(key)) << 4) + (d & 7) * 2));
              }
              typedef __attribute__((__vector_size__(8 * sizeof(short)))) short i16x8;
              const i16x8 both = __builtin_shufflevector(part[0], part[1], 0, 1, 2, 3, 4, 5, 6, 7);
              o[hd][db] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, both), pf[cc], o[hd][db], 0, 0, 0);
            }
        }
        l_run[hd] = lsum;
      }
    }
  };

  // Two (KG) blocks per step: the step's loads refill the stages the previous step read (every wavefront has left them),
  // have the step's arithmetic to land behind, and are met with one wait + barrier.
  for (int i = 0; i < nblk; i += STEP) {
    issue_step(i + STEP);
    if constexpr (KG == 1) {
      process(blk_lo + i, i & (NSTG - 1));
      if (i + 1 < nblk) process(blk_lo + i + 1, (i + 1) & (NSTG - 1));
    } else {
      if (i + kgrp < nblk) process(blk_lo + i + kgrp, (i + kgrp) & (NSTG - 1));
    }
    wait_and_meet();
  }

  // ---- the sink joins the denominator; normalise. A lane holds 8-byte runs of ONE query's row, so storing from here
  // would be 64 scattered 8-byte writes per instruction (measured: ~3 us of a workgroup's life). The wavefront's
  // 32 x (NH x 64) tile goes through its own patch of the now idle stages instead and leaves as whole 128-byte rows.
  constexpr int OROW = NH * 128 + 16;            // patch row: the NH heads of a query + padding (2-way conflicts at most)
  unsigned char* patch = smem + (KG == 1 ? wave : wave % QG) * (32 * OROW);
  if constexpr (KG == 1) {
#pragma unroll
    for (int hd = 0; hd < NH; ++hd) {
      const float l_tot = l_run[hd] + other_half(l_run[hd], h);
      const float sk = a.sinks ? static_cast<float>(a.sinks[head0 + hd]) * kLog2e : 0.f;
      const float m_f = fmaxf(m_run[hd], sk);
      const float so = __builtin_amdgcn_exp2f(m_run[hd] - m_f);
      const float inv = so / fmaf(l_tot, so, __builtin_amdgcn_exp2f(sk - m_f));
#pragma unroll
      for (int db = 0; db < 2; ++db)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          bf16x4 w;
#pragma unroll
          for (int i = 0; i < 4; ++i) w[i] = static_cast<bf16>(o[hd][db][4 * j + i] * inv);
          *reinterpret_cast<bf16x4*>(patch + l31 * OROW + hd * 128 + (db * 32 + 8 * j + 4 * h) * 2) = w;
        }
    }
  } else {
    // The key groups' shares of a query group meet in the idle stages: the accumulator as it is (32 values of 64 lanes), the
    // running maximum and the sum. Wavefront kgrp adds 32 / KG of the 32 values up.
    constexpr int SHARE = 34 * 64;                 // floats of a wavefront
    constexpr int RPG = 32 / KG;
    float* const shares = reinterpret_cast<float*>(smem + QG * 32 * OROW);
    float* const mine = shares + wave * SHARE + lane;
#pragma unroll
    for (int r = 0; r < 32; ++r) mine[r * 64] = o[0][r >> 4][r & 15];
    mine[32 * 64] = m_run[0];
    mine[33 * 64] = l_run[0] + other_half(l_run[0], h);
    __syncthreads();
    const float* const from = shares + (wave % QG) * SHARE + lane;   // key group k: + k * QG * SHARE
    const float sk = a.sinks ? static_cast<float>(a.sinks[head0]) * kLog2e : 0.f;
    float m_f = sk;
#pragma unroll
    for (int k = 0; k < KG; ++k) m_f = fmaxf(m_f, from[k * QG * SHARE + 32 * 64]);
    float den = __builtin_amdgcn_exp2f(sk - m_f);
    float v[RPG] = {};
#pragma unroll
    for (int k = 0; k < KG; ++k) {
      const float* const p = from + k * QG * SHARE;
      const float f = __builtin_amdgcn_exp2f(p[32 * 64] - m_f);      // a group without a visible key: exp2(-inf) = 0
      den = fmaf(p[33 * 64], f, den);
#pragma unroll
      for (int r = 0; r < RPG; ++r) v[r] = fmaf(p[(RPG * kgrp + r) * 64], f, v[r]);
    }
    const float inv = 1.f / den;
#pragma unroll
    for (int r = 0; r < RPG; r += 4) {
      const int rr = RPG * kgrp + r, db = rr >> 4, j = rr >> 2 & 3;
      bf16x4 w;
#pragma unroll
      for (int i = 0; i < 4; ++i) w[i] = static_cast<bf16>(v[r + i] * inv);
      *reinterpret_cast<bf16x4*>(patch + l31 * OROW + (db * 32 + 8 * j + 4 * h) * 2) = w;
    }
    __syncthreads();
  }
  // 16-byte chunks in row-major order: eight lanes per 128-byte head row, NH x 8 per query
  bf16* ob = a.out + b * a.out_bs + head0 * 64;
#pragma unroll
  for (int it = 0; it < NH * 4 / KG; ++it) {
    const int idx = (it * KG + kgrp) * 64 + lane;
    const int row = idx / (NH * 8), ch = idx % (NH * 8);
    const bf16x8 w = *reinterpret_cast<const bf16x8*>(patch + row * OROW + ch * 16);
    if (qw0 + row < a.n_q) *reinterpret_cast<bf16x8*>(ob + static_cast<int64_t>(qw0 + row) * a.out_ts + ch * 8) = w;
  }
}

// Long walks that are not shared out: the same tiles, taken as chunks of 32 keys x one head so that the matrix cores and the
// vector ALU work at the same time.
//
// A wavefront's chunk is 4 MFMAs of S^T, 16 exponentials per lane, 4 MFMAs of O^T and the row sums. One after the other they
// leave the matrix cores idle during the exponentials and the vector ALU idle during the MFMAs, and two wavefronts per SIMD
// do not make up for it (the kernel above, 8192 queries: matrix cores busy 44 % of 1.17 M cycles, vector ALU 64 %). Here the
// interval of chunk i issues, in turn, S^T of chunk i + 1, the exponentials of chunk i and P.V of chunk i - 1, across blocks as
// well: an MFMA, then the two to five vector instructions that fit behind its 32 cycles.
//   * No maximum is taken of a block, except of a wavefront's first one. The weights of a chunk are computed from the running
//     reference as it stands, and one OR over their bf16 bits tells whether any has reached 2 (or is no number): only then the
//     maximum is taken, the reference raised and the chunk's weights computed again. The reference lies 2^7 above the maximum
//     it was raised to, so that this is the same "more than 2^8 above" as there.
//   * The row sums are MFMAs as well (v_dot2c_f32_bf16 does not run beside an MFMA: 64 of them next to 16 MFMAs of another
//     wavefront take 812 cycles, apart 512 and 288): 4 x 4 x 4 ones of ones and the weights, which leave a lane the sum of its
//     own four (16 x 16 x 32 ones do eight times the multiplications: 8192 queries 526 us, so 523, without any sums 496).
//   * One barrier per block, in the middle of the block before: four stages, up to three blocks in flight. What happens rarely
//     is laid out behind the loop, so that the loop's branches fall through.
// 8192 queries 564 -> 523 us (on other GPUs 571 -> 550; 1.17 M -> 0.95 M cycles, but the clock under this load falls from 2.08 to 1.8 GHz:
// what bounds it now is power, and 345 cycles of issue per chunk, of which 16 x 13 are the exponentials and their arguments), 2048 queries
// 50.5 - 53 -> 46.6 - 49.6, 2000 behind 2000 116 -> 107, 600 behind 2000 49 -> 40, 777 queries 15.9 -> 13.6. Windows of up to 321 keys and caches
// of up to six blocks stay with the kernel above: what short walks pay is the first and the last block, and that one is lighter there (8192 queries,
// window of 128: 65 us here, 50 there).
template <int NH, int QG, int NW>
__global__ __launch_bounds__(NW * 64, NW / 2) void attn_prefill_chunks_kernel(AttnPrefillArgs a) {
  constexpr int PBM = 32 * QG;                    // queries per workgroup
  constexpr int HS = NW / QG;                     // head sets
  constexpr int NC = 2 * NH;                      // chunks of a block
  constexpr int DPT = 16 / NW;                    // global->LDS load instructions (1 KB each) per wavefront and block
  static_assert(HS * QG == NW, "wavefronts of a workgroup");
  extern __shared__ __align__(1024) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l31 = lane & 31, h = lane >> 5;

  // workgroup -> (kv head, head sub-group, batch row, query tile); kv head fastest. Long tiles go first; when the whole
  // launch is resident at once (two workgroups per CU), the second workgroup of each CU is taken in the opposite
  // order, so a CU that got a long tile gets a short one next to it.
  const int nsub = a.group / (NH * HS);
  const int ntiles = (a.n_q + PBM - 1) / PBM;
  unsigned id = blockIdx.x;
  const int kvh = id % a.n_kv_heads;
  id /= a.n_kv_heads;
  {
    const unsigned per_round = 256 / (a.n_kv_heads < 256 ? a.n_kv_heads : 256);      // first workgroups of the CUs, per KV head
    const unsigned n = gridDim.x / a.n_kv_heads;
    if (per_round > 0 && n <= 2 * per_round && id >= per_round) id = n + per_round - 1 - id;
  }
  const int sub = id % nsub;
  id /= nsub;
  const int b = id % a.batch;
  id /= a.batch;
  const int tile = ntiles - 1 - static_cast<int>(id);
  const int head0 = kvh * a.group + (sub * HS + wave / QG) * NH;

  // ---- Q fragments (B operand: lane = query, 8 d per half-wavefront and k16 step), requested before the start
  // position is read: their addresses do not depend on it, so they travel while that (dependent) load is on its way
  const int q0 = tile * PBM;
  const int qw0 = q0 + (wave % QG) * 32;   // the wavefront's first query
  bf16x8 qf[NH][4];
  {
    int qrow = qw0 + l31;
    qrow = qrow < a.n_q ? qrow : a.n_q - 1;
    const bf16* qp = a.q + b * a.q_bs + static_cast<int64_t>(qrow) * a.q_ts + head0 * 64 + h * 8;
#pragma unroll
    for (int hd = 0; hd < NH; ++hd)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) qf[hd][kk] = *reinterpret_cast<const bf16x8*>(qp + hd * 64 + kk * 16);
  }

  const int start = a.start_is_i64 ? static_cast<int>(*reinterpret_cast<const int64_t*>(a.start_q)) : *reinterpret_cast<const int*>(a.start_q);
  const int p0 = start + qw0;              // the position of the wavefront's first query
  const int q_end = q0 + PBM < a.n_q ? q0 + PBM : a.n_q;
  int kv_hi = start + q_end < a.n_kv_ctx ? start + q_end : a.n_kv_ctx;       // keys the tile's last query sees (exclusive)
  kv_hi = kv_hi > 0 ? kv_hi : 0;
  int kv_lo = a.window > 0 ? start + q0 - a.window + 1 : 0;
  kv_lo = kv_lo > 0 ? kv_lo : 0;
  kv_lo = kv_lo < kv_hi ? kv_lo : kv_hi;
  const int blk_lo = kv_lo / PBN, blk_hi = (kv_hi + PBN - 1) / PBN;
  const int nblk = blk_hi - blk_lo;
  const int key_max = kv_hi - 1;           // rows beyond it are never visible and may hold anything: not loaded
  // the blocks (counted from blk_lo) of which any of the wavefront's 32 queries sees a key: one run of them
  int w_hi = p0 + 31 >= 0 ? (p0 + 31) / PBN + 1 - blk_lo : 0;
  w_hi = w_hi < nblk ? w_hi : nblk;
  w_hi = w_hi > 0 ? w_hi : 0;
  int w_lo = a.window > 0 && p0 - a.window + 1 > 0 ? (p0 - a.window + 1) / PBN - blk_lo : 0;
  w_lo = w_lo > 0 ? w_lo : 0;
  w_lo = w_lo < w_hi ? w_lo : w_hi;

  // ---- K / V block movers: global_load_lds_dwordx4 (no staging registers, no LDS writes). One instruction fills
  // 1 KB = 8 tile rows, the lanes' 16 bytes landing at M0 + 16 * lane; the swizzle is applied by choosing which chunk of
  // the row a lane fetches. A stage is the K tile followed by the V tile, so a wavefront's DPT instructions all belong
  // to one of the two. A whole block's rows are addressed as a scalar base and 32-bit offsets.
  const int dma_first = wave * DPT;               // the wavefront's first instruction of the block's sixteen: eight of K, eight of V
  const bool dma_v = dma_first >= 8;
  const bf16* const dma_src = (dma_v ? a.v : a.k) + b * a.kv_bs + kvh * 64;
  const bool small_stride = a.kv_ts < (1 << 23);  // 64 rows within 2^30 bytes
  int dma_row[DPT], dma_col[DPT];
  unsigned dma_off[DPT];
#pragma unroll
  for (int j = 0; j < DPT; ++j) {
    const int row = ((dma_first + j) & 7) * 8 + (lane >> 3);
    dma_row[j] = row;
    dma_col[j] = ((lane & 7) ^ (dma_v ? v_swizzle(row) : ((row >> 1) & 7))) * 8;
    dma_off[j] = (static_cast<unsigned>(row) * static_cast<unsigned>(a.kv_ts) + dma_col[j]) * 2;
  }
  const unsigned lds0 = static_cast<unsigned>(reinterpret_cast<uintptr_t>(smem)) + dma_first * 1024;
  auto issue_block = [&](int i) {                 // block i, counted from blk_lo, into stage i & 3
    const int key0 = (blk_lo + i) * PBN;
    const unsigned stage = lds0 + (i & 3) * PSTAGE;
    if (__builtin_expect(key0 + PBN - 1 <= key_max && small_stride, 1)) {         // no row of the block lies beyond the last visible key
      const bf16* const base = dma_src + static_cast<int64_t>(key0) * a.kv_ts;
#pragma unroll
      for (int j = 0; j < DPT; ++j)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(stage + j * 1024), "v"(dma_off[j]), "s"(base) : "memory", "m0");
    } else {
#pragma unroll
      for (int j = 0; j < DPT; ++j) {
        int key = key0 + dma_row[j];
        key = key < key_max ? key : key_max;
        const bf16* const g = dma_src + static_cast<int64_t>(key) * a.kv_ts + dma_col[j];
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off" ::"s"(stage + j * 1024), "v"(g) : "memory", "m0");
      }
    }
  };
  // In the middle of block i (counted from blk_lo): block i + 1 has landed for every wavefront, and every wavefront has read the
  // last of block i - 1, whose stage takes block i + 3.
  auto advance = [&](int i) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(DPT) : "memory");
    if (__builtin_expect(i + 2 >= nblk, 0)) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    asm volatile("s_barrier" ::: "memory");
    if (__builtin_expect(i + 3 < nblk, 1)) issue_block(i + 3);
  };

  // K fragment (A operand of S^T): lane = key l31 of a 32-key half, 16 bytes at d = kk*16 + h*8
  unsigned k_off[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) k_off[kk] = l31 * 128 + (((kk * 2 + h) ^ ((l31 >> 1) & 7)) << 4);      // + 4096 * kb
  // V^T fragment (A operand of O^T): lane = d; the transposing read wants from lane j of each 16 the address of
  // four d (quad j % 4 of the lane group's 16) of key j / 4 of the four keys this half-wavefront takes
  unsigned v_off[2][2];                                                // [u][db]: + 4096 * kb + 2048 * cc
#pragma unroll
  for (int u = 0; u < 2; ++u)
#pragma unroll
    for (int db = 0; db < 2; ++db) {
      const int key = u * 8 + 4 * h + ((lane & 15) >> 2), d = db * 32 + (l31 & 16) + 4 * (lane & 3);
      v_off[u][db] = KT_BYTES + key * 128 + (((d >> 3) ^ v_swizzle(key)) << 4) + (d & 7) * 2;
    }

  // ---- running state: lane = query; the reference (negated) in log2 units of the scaled logits
  const float c = a.sm_scale * kLog2e;
  float neg_ref[NH];
  f32x4 sum[NH];
  f32x16 o[NH][2];
#pragma unroll
  for (int hd = 0; hd < NH; ++hd) {
    neg_ref[hd] = kNoRef;
    sum[hd] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int r = 0; r < 16; ++r) o[hd][db][r] = 0.f;
  }
  const i16x4 ones = {0x3f80, 0x3f80, 0x3f80, 0x3f80};
  float sink[NH];
#pragma unroll
  for (int hd = 0; hd < NH; ++hd) sink[hd] = a.sinks ? static_cast<float>(a.sinks[head0 + hd]) * kLog2e : 0.f;

  for (int i = 0; i < 2 && i < nblk; ++i) issue_block(i);
  {
    // The compiler does not see the direct-to-LDS loads in its count of outstanding loads; were the fragments first
    // used inside the loop, its wait for them there would be "nothing outstanding" and drain the blocks in flight on
    // every step. Pin the wait here, where the first blocks have to land anyway.
#pragma unroll
    for (int hd = 0; hd < NH; ++hd)
#pragma unroll
      for (int kk = 0; kk < 4; ++kk) asm volatile("" : "+v"(qf[hd][kk]));
  }
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  if (2 < nblk) issue_block(2);

  // chunk j's S^T is in s[j & 1], its weights in p[j & 1]
  f32x16 s[2];
  u32x4 p[2][2];
  bf16x8 kf[4], vf[2][2];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      p[j][e] = u32x4{0u, 0u, 0u, 0u};
      vf[j][e] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
    }
  const f32x16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  auto load_k = [&](int i, int kb) __attribute__((always_inline)) {
    const unsigned char* const ks = smem + (i & 3) * PSTAGE + kb * 4096;
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) kf[kk] = *reinterpret_cast<const bf16x8*>(ks + k_off[kk]);
  };
  auto load_v = [&](int i, int kb) __attribute__((always_inline)) {
    const unsigned char* const vs = smem + (i & 3) * PSTAGE + kb * 4096;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc)
#pragma unroll
      for (int db = 0; db < 2; ++db) {
        i16x4 part[2];
#pragma unroll
        for (int u = 0; u < 2; ++u)
          part[u] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(vs + cc * 2048 + v_off[u][db]));
        typedef __attribute__((__vector_size__(8 * sizeof(short)))) short i16x8;
        const i16x8 both = __builtin_shufflevector(part[0], part[1], 0, 1, 2, 3, 4, 5, 6, 7);
        vf[cc][db] = __builtin_bit_cast(bf16x8, both);
      }
  };
  auto qk = [&](int hd, f32x16& d, int kk) __attribute__((always_inline)) {
    d = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kf[kk], qf[hd][kk], kk == 0 ? zero : d, 0, 0, 0);
  };
  // O^T[d, query] += V^T[d, keys] . P^T[keys, query] in four, the sum of the rounded weights in two
  auto pv = [&](int hd, const u32x4 (&w)[2], int n) __attribute__((always_inline)) {
    if (n < 4) {
      o[hd][n & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vf[n >> 1][n & 1], __builtin_bit_cast(bf16x8, w[n >> 1]), o[hd][n & 1], 0, 0, 0);
    } else {
      typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned u32x2;
      const u32x2 lo = {w[n - 4][0], w[n - 4][1]}, hi = {w[n - 4][2], w[n - 4][3]};
      sum[hd] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ones, __builtin_bit_cast(i16x4, lo), sum[hd], 0, 0, 0);
      sum[hd] = __builtin_amdgcn_mfma_f32_4x4x4bf16_1k(ones, __builtin_bit_cast(i16x4, hi), sum[hd], 0, 0, 0);
    }
  };
  auto weight = [&](float x, float nr) { return __builtin_amdgcn_exp2f(fmaf(x, c, nr)); };
  auto pack = [](float x, float y) {
    const bf16x2 v = {static_cast<bf16>(x), static_cast<bf16>(y)};
    return __builtin_bit_cast(unsigned, v);
  };
  // the keys of block i that the lane's query does not see: behind the causal diagonal or the end of the keys (1), before the window (2)
  const int upper = p0 + l31 < a.n_kv_ctx - 1 ? p0 + l31 : a.n_kv_ctx - 1, lower = p0 + l31 - a.window + 1;
  auto crossed = [&](int i) {
    const int key0 = (blk_lo + i) * PBN;
    return (key0 + PBN - 1 > p0 || key0 + PBN - 1 >= a.n_kv_ctx ? 1 : 0) | (a.window > 0 && key0 < p0 + 31 - a.window + 1 ? 2 : 0);
  };
  auto mask = [&](f32x16& d, int i, int kb, int crosses) __attribute__((always_inline)) {
    const int key0 = (blk_lo + i) * PBN + kb * 32 + 4 * h;
    const int du = upper - key0, dl = lower - key0;
    if (crosses & 1) {
#pragma unroll
      for (int r = 0; r < 16; ++r) d[r] = 8 * (r >> 2) + (r & 3) <= du ? d[r] : -INFINITY;
    }
    if (crosses & 2) {
#pragma unroll
      for (int r = 0; r < 16; ++r) d[r] = 8 * (r >> 2) + (r & 3) >= dl ? d[r] : -INFINITY;
    }
  };
  auto chunk = [&](int i, int crosses, auto tag) __attribute__((always_inline)) {
    constexpr int C = decltype(tag)::value;
    constexpr int kb = C / NH, hd = C % NH, cur = C & 1, nxt = cur ^ 1;
    constexpr int nhd = (C + 1) % NH, phd = (C + NC - 1) % NH, pkb = (C + NC - 1) % NC / NH;
    if constexpr (phd == 0 && C > 0) {
      load_v(i, pkb);
    } else if constexpr (phd == 0) {             // one head: the half of the block before
      if (i > w_lo) load_v(i - 1, pkb);
    }
    if (__builtin_expect(crosses != 0, 0)) mask(s[cur], i, kb, crosses);
    float e[2][2];
    auto pair_exp = [&](int m) __attribute__((always_inline)) {
      e[m & 1][0] = weight(s[cur][2 * m], neg_ref[hd]);
      e[m & 1][1] = weight(s[cur][2 * m + 1], neg_ref[hd]);
    };
    auto pair_pack = [&](int m) __attribute__((always_inline)) { p[cur][m >> 2][m & 3] = pack(e[m & 1][0], e[m & 1][1]); };
#pragma unroll
    for (int m = 0; m < 4; ++m) {
      qk(nhd, s[nxt], m);
      pair_exp(m);
      if (m > 0) pair_pack(m - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (C == NC - 2) {
      asm volatile("" : "+v"(e[0][0]), "+v"(e[0][1]), "+v"(e[1][0]), "+v"(e[1][1]), "+v"(p[cur][0]));     // not moved behind the barrier
      advance(i);
    }
    if constexpr ((C + 2) % NH == 0) load_k(C + 2 >= NC ? i + 1 : i, (C + 2) % NC / NH);
#pragma unroll
    for (int m = 4; m < 8; ++m) {
      pv(phd, p[nxt], m - 4);
      pair_exp(m);
      pair_pack(m - 1);
      __builtin_amdgcn_sched_barrier(0);
    }
    pv(phd, p[nxt], 4);
    pair_pack(7);
    pv(phd, p[nxt], 5);
    unsigned any = 0;
#pragma unroll
    for (int m = 0; m < 8; ++m) any |= p[cur][m >> 2][m & 3];
    if (__builtin_expect(__builtin_amdgcn_ballot_w64((any & 0x40004000u) != 0) != 0, 0)) {          // a weight of 2 or more, or no number
      float t = -INFINITY;
#pragma unroll
      for (int r = 0; r < 16; ++r) t = fmaxf(t, s[cur][r]);
      t = fmaxf(t, other_half(t, h)) * c;
      const float ref = -neg_ref[hd];
      const bool raise = t > ref + (kRaise - kLift);                           // false while nothing is visible (t is -inf)
      const float moved = raise ? t + kLift : ref;
      const float alpha = raise ? __builtin_amdgcn_exp2f(ref - moved) : 1.f;   // from no reference: 0
      neg_ref[hd] = -moved;
      // (pinned as whole registers on both sides: the copies that the compiler makes to join the two paths stay in this one)
      auto scale = [&](auto& v, int n) __attribute__((always_inline)) {
        asm volatile("" : "+v"(v));
#pragma unroll
        for (int r = 0; r < n; ++r) v[r] *= alpha;
        asm volatile("" : "+v"(v));
      };
      scale(sum[hd], 4);
      scale(o[hd][0], 16);
      scale(o[hd][1], 16);
#pragma unroll
      for (int m = 0; m < 8; ++m) p[cur][m >> 2][m & 3] = pack(weight(s[cur][2 * m], neg_ref[hd]), weight(s[cur][2 * m + 1], neg_ref[hd]));
      asm volatile("" : "+v"(p[cur][0]), "+v"(p[cur][1]));
    }
  };

  // Blocks that only the other wavefronts of the workgroup need, the wavefront's own, and again the others'.
  int i = 0;
  for (; i < w_lo; ++i) advance(i);
  if (w_lo < w_hi) {
    // the reference: the maximum of the first block
#pragma unroll
    for (int hd = 0; hd < NH; ++hd) {
      float t = -INFINITY;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        load_k(i, kb);
#pragma unroll
        for (int kk = 0; kk < 4; ++kk) qk(hd, s[kb], kk);
      }
      const int crosses = crossed(i);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        if (crosses != 0) mask(s[kb], i, kb, crosses);
#pragma unroll
        for (int r = 0; r < 16; ++r) t = fmaxf(t, s[kb][r]);
      }
      t = fmaxf(t, other_half(t, h)) * c;
      neg_ref[hd] = t > -kNoRef ? -(t + kLift) : kNoRef;
    }
    load_k(i, 0);
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) qk(0, s[0], kk);
    if constexpr (NH == 1) load_k(i, 1);
    for (; i < w_hi; ++i) {
      const int crosses = crossed(i);
      chunk(i, crosses, std::integral_constant<int, 0>{});
      chunk(i, crosses, std::integral_constant<int, 1>{});
      if constexpr (NH == 2) {
        chunk(i, crosses, std::integral_constant<int, 2>{});
        chunk(i, crosses, std::integral_constant<int, 3>{});
      }
    }
    if constexpr (NH == 1) load_v(i - 1, 1);      // P.V of the last chunk
#pragma unroll
    for (int n = 0; n < 6; ++n) pv(NH - 1, p[1], n);
  }
  for (; i < nblk; ++i) advance(i);
  __syncthreads();

  // ---- the sink joins the denominator; normalise. A lane holds 8-byte runs of ONE query's row, so storing from here
  // would be 64 scattered 8-byte writes per instruction (measured: ~3 us of a workgroup's life). The wavefront's
  // 32 x (NH x 64) tile goes through its own patch of the now idle stages instead and leaves as whole 128-byte rows.
  constexpr int OROW = NH * 128 + 16;            // patch row: the NH heads of a query + padding (2-way conflicts at most)
  unsigned char* patch = smem + wave * (32 * OROW);
#pragma unroll
  for (int hd = 0; hd < NH; ++hd) {
    const float ref = neg_ref[hd] == kNoRef ? -INFINITY : -neg_ref[hd];
    const float sk = sink[hd];
    const float m_f = fmaxf(ref, sk);
    const float so = __builtin_amdgcn_exp2f(ref - m_f);
    const float inv = so / fmaf(sum[hd][0] + other_half(sum[hd][0], h), so, __builtin_amdgcn_exp2f(sk - m_f));
#pragma unroll
    for (int db = 0; db < 2; ++db)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        bf16x4 w;
#pragma unroll
        for (int e = 0; e < 4; ++e) w[e] = static_cast<bf16>(o[hd][db][4 * j + e] * inv);
        *reinterpret_cast<bf16x4*>(patch + l31 * OROW + hd * 128 + (db * 32 + 8 * j + 4 * h) * 2) = w;
      }
  }
  // 16-byte chunks in row-major order: eight lanes per 128-byte head row, NH x 8 per query
  bf16* ob = a.out + b * a.out_bs + head0 * 64;
#pragma unroll
  for (int it = 0; it < NH * 4; ++it) {
    const int idx = it * 64 + lane;
    const int row = idx / (NH * 8), ch = idx % (NH * 8);
    const bf16x8 w = *reinterpret_cast<const bf16x8*>(patch + row * OROW + ch * 16);
    if (qw0 + row < a.n_q) *reinterpret_cast<bf16x8*>(ob + static_cast<int64_t>(qw0 + row) * a.out_ts + ch * 8) = w;
  }
}

}  // namespace tllm

using namespace tllm;

template <int NH, int QG, int KG, int NW>
static int launch_prefill(const AttnPrefillArgs& a, hipStream_t st) {
  constexpr int SMEM = 2 * (KG == 1 ? 2 : KG) * PSTAGE, HS = NW / (QG * KG);
  static_assert(KG == 1 || QG * 32 * (128 + 16) + NW * 34 * 256 <= SMEM, "the key groups' shares fit the stages");
  static_assert(KG > 1 || NW * 32 * (NH * 128 + 16) <= SMEM, "the output patches fit the stages");
  static std::atomic<uint64_t> done{0};
  const hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(attn_prefill_kernel<NH, QG, KG, NW>), SMEM, done);
  TLLM_REQUIRE(e == hipSuccess, TLLM_E_LAUNCH, "attention_prefill: cannot raise LDS limit: %s", hipGetErrorString(e));
  const int64_t wgs = static_cast<int64_t>((a.n_q + 32 * QG - 1) / (32 * QG)) * a.batch * a.n_kv_heads * (a.group / (NH * HS));
  TLLM_REQUIRE(wgs < (1ll << 31), TLLM_E_SHAPE, "attention_prefill: %lld workgroups are too many for one launch", (long long)wgs);
  hipLaunchKernelGGL((attn_prefill_kernel<NH, QG, KG, NW>), dim3((unsigned)wgs), dim3(NW * 64), SMEM, st, a);
  return check_launch("attention_prefill");
}

template <int NH, int QG, int NW>
static int launch_prefill_chunks(const AttnPrefillArgs& a, hipStream_t st) {
  constexpr int SMEM = 4 * PSTAGE, HS = NW / QG;
  static_assert(NW * 32 * (NH * 128 + 16) <= SMEM, "the output patches fit the stages");
  static std::atomic<uint64_t> done{0};
  const hipError_t e = raise_lds_limit(reinterpret_cast<const void*>(attn_prefill_chunks_kernel<NH, QG, NW>), SMEM, done);
  TLLM_REQUIRE(e == hipSuccess, TLLM_E_LAUNCH, "attention_prefill: cannot raise LDS limit: %s", hipGetErrorString(e));
  const int64_t wgs = static_cast<int64_t>((a.n_q + 32 * QG - 1) / (32 * QG)) * a.batch * a.n_kv_heads * (a.group / (NH * HS));
  TLLM_REQUIRE(wgs < (1ll << 31), TLLM_E_SHAPE, "attention_prefill: %lld workgroups are too many for one launch", (long long)wgs);
  hipLaunchKernelGGL((attn_prefill_chunks_kernel<NH, QG, NW>), dim3((unsigned)wgs), dim3(NW * 64), SMEM, st, a);
  return check_launch("attention_prefill");
}

// Blocks that the longest walk of 64 queries over the keys can have: the host knows the size of the cache and the window, not where in the
// cache the queries start (and counts from an aligned start).
static int64_t longest_walk(int64_t n_kv_ctx, int window) {
  const int64_t all = (n_kv_ctx + PBN - 1) / PBN, seen = (static_cast<int64_t>(window) + 126) / PBN;
  return window > 0 && seen < all ? seen : all;
}

// Workgroup shape, by how many workgroups the launch has and how long they walk. When 64 queries x 1 head are at most two
// workgroups per CU, the wavefronts share the key blocks out: two groups of two wavefronts, or four (one workgroup of eight
// wavefronts per CU), us before -> so:
//   97 queries behind 1500 keys 27.0 -> 16.1 (two groups 18.3), with a window of 128 9.3 -> 6.9; 16 behind 4000 58.3 -> 29.9;
//   256 behind 2000 37.4 -> 20.3 (23.8); 400 queries 11.3 -> 9.7; 500 behind 1000 27.4 -> 21.3; 512 behind 4000 67.9 -> 56.1
//   (from three workgroups per CU on the longer walk is hidden by the others: 777 queries 17.8, shared out 19.1).
// A walk has to be long enough to pay for the meeting at its end: more than one block (16 or 64 queries alone 5.5 us, shared
// out 6.1; two blocks, 97 queries, 6.6 and 6.3), and at two workgroups per CU more than three (eight prompts of 64 6.2 and
// 7.5, four of 128 6.9 and 7.6, window of 128: 400 queries 8.2 and 9.4, 512 8.3 and 9.5; five blocks, 300 queries, 9.4 and 8.9).
extern "C" int tllm_attention_prefill_key_groups(int64_t batch, int64_t n_q, int64_t n_kv_ctx, int n_kv_heads, int group, int window) {
  const int64_t wgs64 = (n_q + 63) / 64 * batch * n_kv_heads * group;
  const int64_t span = window > 0 && window < n_kv_ctx - n_q ? n_q + window : n_kv_ctx;     // most keys there can be to visit
  const int64_t walk = longest_walk(n_kv_ctx, window);
  if (wgs64 <= 256 && span > 192) return 4;
  return wgs64 <= 512 && walk > (wgs64 <= 256 ? 1 : 3) ? 2 : 1;
}

// Otherwise 64 queries x 4 heads with two heads per wavefront, or, where those are too few workgroups, 64 queries x 2 heads with
// one per wavefront: twice the workgroups, and the longest of them -- it sets the time of a small launch -- takes about half as
// long per key block. The line, with few / many heads in us. Short walks (window of 128): 2 x 500 queries (256 of the
// workgroups with four heads) 10.4 / 11.1, 1100 (288) 13.6 / 13.0, 2048 18.4 / 16.4, 8192 60.7 / 50.1. Five or six blocks: 3 x 333
// (288) 12.8 / 14.3, 4 x 384 (384) 16.8 / 15.9, 5 x 300 (400) 15.7 / 14.6. Walks in chunks of up to 12 blocks: 2 x 600 (320) 17.7 /
// 19.9, 2 x 700 (352) 20.7 / 21.9, 3 x 450 (384) 18.2 / 17.9, with 300 keys before 25.9 / 26.8; longer ones: 1536 (384) 31.1 / 34.9, 1900 (480) 43.6 /
// 43.7, with 300 keys before 54.2 / 51.9, 4096 156 / 147. (128 queries x 2 heads, which they replace, are never ahead: an 8192 window 55.8 and 50.1, 3000
// queries 90.9 and 88.1.) Groups that are no multiple of four take 128 x 2, odd ones 128 x 1.
// In chunks where the cache has more than six blocks, which a prompt may not walk. Of 294 batches of 1 - 16 prompts of 64 - 1300 tokens behind
// 0 - 1000, in caches of their own length and of 4096, what is chosen here takes 0.91 of the time it took without chunks and with 128 queries x 2
// heads, in the mean; one head per wavefront in chunks takes 0.94 - 0.975 of the other kernel's where walks are three to six blocks (4 x 300 in a
// cache of 4096 15.3 / 14.4, 2 x 384 11.8 / 10.8, 8 x 128 9.07 / 8.82). Behind by more than 1 % are 3 x 333 (13.8 / 14.0), 3 x 384 (14.3 / 14.6), 2 x 600 (17.0 / 17.7) and 2 x 700 (20.2 / 20.7; with 100 keys before 23.9 / 22.3 and
// 26.6 / 24.4), and with five heads 8 x 128 (9.16 / 9.34).
namespace {
struct PrefillShape {
  int queries, heads, key_groups;      // of a workgroup
  bool chunks;
};

PrefillShape prefill_shape(int64_t batch, int64_t n_q, int64_t n_kv_ctx, int n_kv_heads, int group, int window) {
  const int key_groups = tllm_attention_prefill_key_groups(batch, n_q, n_kv_ctx, n_kv_heads, group, window);
  if (key_groups > 1) return {64, 1, key_groups, false};
  const int64_t walk = longest_walk(n_kv_ctx, window);
  const bool chunks = walk > 6;
  if (group % 2 != 0) return {128, 1, 1, chunks};
  const int64_t wgs4 = (n_q + 63) / 64 * batch * n_kv_heads * group / 4;
  if (wgs4 < (chunks ? (walk <= 12 ? 368 : 432) : (walk <= 4 ? 272 : 320))) return {64, 2, 1, chunks};
  return group % 4 == 0 ? PrefillShape{64, 4, 1, chunks} : PrefillShape{128, 2, 1, chunks};
}
}  // namespace

extern "C" int tllm_attention_prefill_shape(int64_t batch, int64_t n_q, int64_t n_kv_ctx, int n_kv_heads, int group, int window) {
  if (batch < 1 || n_q < 1 || n_kv_ctx < 1 || n_kv_heads < 1 || group < 1 || window < 0) return 0;
  const PrefillShape p = prefill_shape(batch, n_q, n_kv_ctx, n_kv_heads, group, window);
  return (p.chunks ? 1 << 24 : 0) | p.queries << 16 | p.heads << 8 | p.key_groups;
}

extern "C" int tllm_attention_prefill_bf16(const void* q, const void* k, const void* v, const void* sinks, void* out, int64_t q_batch_stride,
                                           int64_t q_token_stride, int64_t out_batch_stride, int64_t out_token_stride,
                                           int64_t kv_batch_stride, int64_t kv_token_stride, int64_t batch, int64_t n_q, int64_t n_kv_ctx,
                                           int n_kv_heads, int group, int head_dim, float sm_scale, int window, const void* start_q,
                                           int start_q_is_i64, void* stream) {
  TLLM_REQUIRE(batch >= 0 && n_q >= 0 && n_kv_ctx >= 1 && n_kv_heads >= 1, TLLM_E_SHAPE,
               "attention_prefill: batch %lld, n_q %lld, n_kv_ctx %lld, n_kv_heads %d", (long long)batch, (long long)n_q, (long long)n_kv_ctx,
               n_kv_heads);
  TLLM_REQUIRE(n_kv_ctx < (1ll << 30) && n_q < (1ll << 30), TLLM_E_SHAPE, "attention_prefill: n_q %lld / n_kv_ctx %lld too large",
               (long long)n_q, (long long)n_kv_ctx);
  TLLM_REQUIRE(head_dim == 64, TLLM_E_SHAPE, "attention_prefill: head_dim %d (only 64 is built)", head_dim);
  TLLM_REQUIRE(group >= 1 && group <= 64, TLLM_E_SHAPE, "attention_prefill: %d query heads per KV head (1..64)", group);
  TLLM_REQUIRE(window >= 0, TLLM_E_ARG, "attention_prefill: window %d", window);
  TLLM_REQUIRE(sm_scale > 0.f, TLLM_E_ARG, "attention_prefill: sm_scale %g must be positive", (double)sm_scale);
  if (batch == 0 || n_q == 0) return TLLM_OK;
  TLLM_REQUIRE(q && k && v && out && start_q, TLLM_E_ARG, "attention_prefill: q, k, v, out and start_q must not be NULL");
  const int64_t n_heads = static_cast<int64_t>(n_kv_heads) * group;
  TLLM_REQUIRE(aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out) && q_batch_stride % 8 == 0 && q_token_stride % 8 == 0 &&
                   out_batch_stride % 8 == 0 && out_token_stride % 8 == 0 && kv_batch_stride % 8 == 0 && kv_token_stride % 8 == 0,
               TLLM_E_ALIGN, "attention_prefill: q, k, v, out must be 16-byte aligned with strides that are multiples of 8 elements");
  TLLM_REQUIRE(q_token_stride >= n_heads * 64 && out_token_stride >= n_heads * 64, TLLM_E_ARG,
               "attention_prefill: q / out token stride < n_heads * 64");
  TLLM_REQUIRE(kv_token_stride >= static_cast<int64_t>(n_kv_heads) * 64, TLLM_E_ARG, "attention_prefill: kv_token_stride < n_kv_heads * 64");
  AttnPrefillArgs a{};
  a.q = (const bf16*)q;
  a.k = (const bf16*)k;
  a.v = (const bf16*)v;
  a.sinks = (const bf16*)sinks;
  a.out = (bf16*)out;
  a.start_q = start_q;
  a.start_is_i64 = start_q_is_i64;
  a.q_bs = q_batch_stride;
  a.q_ts = q_token_stride;
  a.out_bs = out_batch_stride;
  a.out_ts = out_token_stride;
  a.kv_bs = kv_batch_stride;
  a.kv_ts = kv_token_stride;
  a.batch = (int)batch;
  a.n_q = (int)n_q;
  a.n_kv_ctx = (int)n_kv_ctx;
  a.n_kv_heads = n_kv_heads;
  a.group = group;
  a.window = window;
  a.sm_scale = sm_scale;
  const int64_t wgs128 = (n_q + 127) / 128 * batch * n_kv_heads * (group % 2 == 0 ? group / 2 : group);
  TLLM_REQUIRE(batch < (1ll << 24) && wgs128 < (1ll << 31), TLLM_E_SHAPE, "attention_prefill: %lld workgroups are too many for one launch", (long long)wgs128);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const PrefillShape p = prefill_shape(batch, n_q, n_kv_ctx, n_kv_heads, group, window);
  if (p.key_groups == 4) return launch_prefill<1, 2, 4, 8>(a, st);
  if (p.key_groups == 2) return launch_prefill<1, 2, 2, 4>(a, st);
  if (p.heads == 1) return p.chunks ? launch_prefill_chunks<1, 4, 4>(a, st) : launch_prefill<1, 4, 1, 4>(a, st);
  if (p.heads == 4) return p.chunks ? launch_prefill_chunks<2, 2, 4>(a, st) : launch_prefill<2, 2, 1, 4>(a, st);
  if (p.queries == 64) return p.chunks ? launch_prefill_chunks<1, 2, 4>(a, st) : launch_prefill<1, 2, 1, 4>(a, st);
  return p.chunks ? launch_prefill_chunks<2, 4, 4>(a, st) : launch_prefill<2, 4, 1, 4>(a, st);
}
