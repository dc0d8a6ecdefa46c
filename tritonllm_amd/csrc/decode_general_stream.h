// The weight stream of the general-shape decode kernels (decode_general.hip): sixteen weight rows times up to XR
// activation rows over any K that is a multiple of 32, on v_mfma_f32_16x16x32_bf16 with the weight rows on M.
//
// What bounds it is how many bytes of the weight are in flight: each CU's share of HBM is ~28 GB/s, two microseconds
// away. NS = 4, 2 or 1 streaming wavefronts deal K by phase -- in phase p wavefront w takes the 128 K (fp8 weight: 256 K) behind
// (NS p + w) * 128, so that four ask for 1 KB contiguous of every row at a time -- and every operand goes from global
// memory straight into LDS (global_load_lds_dwordx4) through a ring of two phases that belongs to the wavefront alone: no
// barrier, no staging registers, and no wavefront waits for another one's loads. Two phases for each of four wavefronts are 48
// KB (fp8 weight or sixteen rows: 64-96), so that two or three workgroups share a CU and a grid that does not divide by 256 (4096
// wide with 80 heads: 320 workgroups) leaves no CU idle early. Measured at hidden 4096, 80 heads of 64, 8 rows: four
// wavefronts with two phases 11.0 us, three 11.1, four (one workgroup per CU) 13.0; eight wavefronts 12.3. The kernel
// before -- a wavefront per workgroup, loads through registers and an LDS patch -- took 14.7.
// s_waitcnt vmcnt is spelled by hand; the streaming wavefronts issue no other vector load.
#pragma once

#include "common.h"

namespace tllm {

// NS: streaming wavefronts of a workgroup (4, 2 or 1)
template <int XR, bool W8, int NS>
struct DecodeGeneralStream {
  static constexpr int KPH = W8 ? 256 : 128;                // K of a wavefront's phase (both: 256 bytes of a weight row)
  static constexpr int PST = KPH / 32;                      // k32 steps of it
  static constexpr int XROW = KPH * 2;                      // bytes of an activation row's piece
  static constexpr int WBYTES = 16 * 256;                   // one phase of the weight ...
  static constexpr int XBYTES = XR * XROW;                  // ... and of the activations
  static constexpr int WL = WBYTES / 1024, XL = XBYTES / 1024;
  static constexpr int LPP = WL + XL;                       // load instructions per phase
  static constexpr int D = 2;                               // phases resident per wavefront
  static constexpr int REGION = WBYTES + XBYTES;
  // LDS of a wavefront; one that has a single phase needs no second one
  static __host__ __device__ __forceinline__ int wave_lds(int K) { return (K > NS * KPH ? D : 1) * REGION; }

  // k8 group (eight consecutive K) that lane group g = lane / 16 supplies in step st of a phase. Any assignment will do
  // as long as both operands agree; this one is made for the LDS: a 128-bit read is served 16 lanes at a time, lanes 0-7
  // together with 32-39, so groups g and g + 2 must read 16-byte chunks that differ in bit 3 (rows are 256 bytes = all
  // banks apart and XOR-swizzled by the row), and the 64-bit reads of an fp8 row take both halves of one chunk in groups
  // 2 i and 2 i + 1.
  static __device__ __forceinline__ int k8_of(int st, int g) { return 16 * (st >> 2) + 8 * (g >> 1) + 2 * (st & 3) + (g & 1); }

  // The wavefront's share of the sixteen dot products, left as a f32x4 per lane at smem + wave * wave_lds() + lane * 16
  // (lane: activation row lane % 16, tile rows 4 (lane / 16) .. + 3). wbase: first byte of the rows' common base,
  // wrow(i): tile row i's row index behind it (any valid row for rows past the last one).
  template <class WRow>
  static __device__ __forceinline__ void run(unsigned char* smem, int wave, int lane, const unsigned char* xbase, int nvalid,
                                             const unsigned char* wbase, WRow wrow, int K) {
    const int m = lane & 15, g = lane >> 4, mx = m & (XR - 1);
    const unsigned wpitch = static_cast<unsigned>(K) * (W8 ? 1 : 2), xpitch = static_cast<unsigned>(K) * 2;
    unsigned char* my = smem + wave * wave_lds(K);
    const int k0 = wave * KPH;
    const int nph = K > k0 ? (K - k0 + NS * KPH - 1) / (NS * KPH) : 0;
    const bool ragged = (K - k0) % (NS * KPH) != 0 && (K - k0) % (NS * KPH) < KPH;   // the last phase is cut short

    // Load j of the weight: rows 4 j + lane / 16, 16-byte position lane % 16 <- chunk position ^ row. Of the
    // activations: a KB is 1024 / XROW rows, position <- chunk position ^ row likewise.
    unsigned wrow_off[WL], wchunk[WL], xrow_off[XL], xchunk[XL];
#pragma unroll
    for (int j = 0; j < WL; ++j) {
      const int r = 4 * j + (lane >> 4);
      wchunk[j] = static_cast<unsigned>((lane & 15) ^ r) * 16u;
      wrow_off[j] = static_cast<unsigned>(wrow(r)) * wpitch;
    }
    constexpr int XPOS = XROW / 16;                         // 16-byte positions of an activation row's piece
#pragma unroll
    for (int j = 0; j < XL; ++j) {
      const int r = j * (1024 / XROW) + lane / XPOS;
      xchunk[j] = static_cast<unsigned>((lane % XPOS) ^ r) * 16u;
      xrow_off[j] = static_cast<unsigned>(r < nvalid ? r : nvalid - 1) * xpitch;
    }
    // Rows whose pitch is a multiple of 4 KB all begin on the same memory channels: the workgroups of an XCD start in different
    // phases and go round (such a K has no ragged phase). [4096, 4096] at 8 rows 7.95 -> 7.1 us, fp8 6.3 -> 5.8,
    // [4096, 8192] 15.5 -> 12.5; at K = 3072, whose rows spread by themselves, it makes no difference.
    const int rot = wpitch % 4096 == 0 && nph > 0 ? static_cast<int>(blockIdx.x >> 3) % nph : 0;
    auto phase = [&](int pp) { return pp + rot < nph ? pp + rot : pp + rot - nph; };
    auto lds_addr = [](const void* p) { return static_cast<unsigned>(reinterpret_cast<uintptr_t>(p)); };
    auto issue = [&](int pp, int slot) {
      const int p = phase(pp);
      unsigned char* reg = my + slot * REGION;
      const unsigned wk = static_cast<unsigned>(p * NS + wave) * 256u, xk = static_cast<unsigned>(p * NS + wave) * XROW;
      // a chunk behind the row's end re-reads the row's last one (its products are masked)
#pragma unroll
      for (int j = 0; j < XL; ++j) {
        const unsigned at = xk + xchunk[j];
        const unsigned off = xrow_off[j] + (at < xpitch ? at : xpitch - 16u);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_addr(reg + WBYTES + j * 1024)), "v"(off), "s"(xbase)
                     : "memory", "m0");
      }
#pragma unroll
      for (int j = 0; j < WL; ++j) {
        const unsigned at = wk + wchunk[j];
        const unsigned off = wrow_off[j] + (at < wpitch ? at : wpitch - 16u);
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt" ::"s"(lds_addr(reg + j * 1024)), "v"(off), "s"(wbase)
                     : "memory", "m0");
      }
    };
#pragma unroll
    for (int p = 0; p < D; ++p)
      if (p < nph) issue(p, p);

    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    int slot = 0;
    for (int p = 0; p < nph; ++p) {
      const int behind = nph - 1 - p;                       // phases requested after this one: one, or none
      if (behind > 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * LPP) : "memory");
      else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      const unsigned char* wr = my + slot * REGION;
      const unsigned char* xr = wr + WBYTES;
      bf16x8 fw[PST], fx[PST];
#pragma unroll
      for (int st = 0; st < PST; ++st) {
        const int e = k8_of(st, g);
        if constexpr (W8) {
          typedef __attribute__((__vector_size__(2 * sizeof(unsigned)))) unsigned u32x2;
          const u32x2 raw = *reinterpret_cast<const u32x2*>(wr + m * 256 + (((e >> 1) ^ m) << 4) + (e & 1) * 8);
          fw[st] = fp8x8_to_bf16x8(raw[0], raw[1]);
        } else {
          fw[st] = *reinterpret_cast<const bf16x8*>(wr + m * 256 + ((e ^ m) << 4));
        }
        fx[st] = *reinterpret_cast<const bf16x8*>(xr + mx * XROW + ((e ^ mx) << 4));
      }
      // the region is free once its fragments are in registers
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      if (p + D < nph) issue(p + D, slot);
      if (ragged && phase(p) == nph - 1) {
        const int left = (K - (phase(p) * NS + wave) * KPH) >> 3;  // k8 groups that exist
#pragma unroll
        for (int st = 0; st < PST; ++st)
          if (k8_of(st, g) >= left) {
            fw[st] = bf16x8{};
            fx[st] = bf16x8{};
          }
      }
#pragma unroll
      for (int st = 0; st < PST; ++st) acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fw[st], fx[st], acc, 0, 0, 0);
      slot = slot + 1 == D ? 0 : slot + 1;
    }
    // every load of this wavefront has landed (the last wait was for zero), so its LDS is free
    *reinterpret_cast<f32x4*>(my + lane * 16) = acc;
  }

  // Behind the barrier that follows run(): the partial tiles added in a fixed order.
  static __device__ __forceinline__ f32x4 sum(const unsigned char* smem, int lane, int K) {
    f32x4 t[NS];
#pragma unroll
    for (int w = 0; w < NS; ++w) t[w] = *reinterpret_cast<const f32x4*>(smem + w * wave_lds(K) + lane * 16);
    if constexpr (NS == 4) return (t[0] + t[1]) + (t[2] + t[3]);
    else if constexpr (NS == 2) return t[0] + t[1];
    else return t[0];
  }
};

}  // namespace tllm
