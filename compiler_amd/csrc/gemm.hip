// GEMM family on gfx950: bf16/fp16 (fp32 accumulate) and int8 (int32
// accumulate, bit-exact) with a fused epilogue.
//
// Operator semantics: ops/suite/perf/matmul.py:21-37 (Y = A.B, fp32
// accumulator, masked M/N/K edges, store in the output pointer dtype);
// int8 dot family a100c/plan/tiles.py:118-131 (signed operands, modular int32
// accumulator); dequant rule ops/suite/perf/dequantize_matmul.py:29-38
// (per-column scale), here with the per-row A scale as well:
// Y[m,n] = bf16(float(acc[m,n]) * sa[m] * sb[n]).
//
// MFMA kernel (g950_gemm_*_256x256): both operands K-contiguous (A row-major
// [M,K]; B stored as Bt[N,K], i.e. column-major [K,N]).  The `_rb` variants
// (16-bit) read the reference's row-major B[K,N] as it lies, with
// transposing LDS reads (the BROW notes above gemm_mfma16_body).
//   * workgroup tile 256x256, 8 waves (4 x 2, two per SIMD), wave tile
//     64 x 128: 4 x 8 fragments of v_mfma_f32_16x16x32_{bf16,f16} /
//     v_mfma_i32_16x16x64_i8 for whole-slab 16-bit / int8 shapes with
//     M, N >= 256 (gemm_mfma16_body), else 2 x 4 fragments of the 32x32
//     forms; shapes whose 256 x 256 tiles leave CUs idle run 128x128, 64x128
//     or 64x64 tiles in the same kernels (gemm_tile_body; the host picks by
//     measured tile times); the B tile feeds the MFMA A port so each lane ends with four
//     consecutive output columns of one output row
//   * K in slabs of 128 bytes per row (64 bf16 / 128 int8); two LDS stages
//     of 64 KiB (A rows then B rows, 128-byte rows), filled by direct
//     global->LDS 16-byte DMA (global_load_lds_dwordx4) of whole 128-byte
//     lines (measured on MI355X: 64-byte row pieces cost the load path 1.5x
//     per byte); the DMA takes a scalar base plus a fixed 32-bit lane offset
//     and the fragment reads fixed per-lane LDS offsets plus immediates, so
//     the main loop holds MFMAs, LDS reads, DMAs and scalar work only
//   * the eight 16-byte chunks of a 128-byte LDS row are XOR-swizzled with
//     (row >> 1) & 7, so the 32 rows an MFMA operand read touches spread over
//     all 64 banks
//   * per slab: four k-steps; each k-step's MFMAs run with the next k-step's
//     fragment reads (second register set) spread between them, and the
//     slab's DMA is spread over k-step 3 of the previous slab and k-step 0
//     (sched_group_barrier), issued by one wave of each SIMD only, so the
//     other wave's MFMAs fill the matrix core while the DMA wave waits on the
//     load path; one workgroup barrier per slab, before k-step 3
//   * XCD-aware block order: consecutive tiles go to the same XCD (the
//     hardware deals workgroups round-robin over 8 XCDs), grouped 4 tile-rows
//     deep for L2 reuse (4 beat 2, 8, 16 and 32 at 8192^3)
//   * M/N edges: loads clamp the row index (the duplicated rows only feed
//     output rows/cols that are never stored); stores are masked.  K must be a
//     whole number of slabs (host checks), otherwise the general kernel runs.
//
// General kernel (g950_gemm_general): any strides, any K, fp32/fp16/bf16
// inputs (fp32 FMA) or int8 (int32 exact); 64x64 tiles.  It serves the
// layouts no MFMA route takes (unaligned rows, non-unit inner strides) and
// the no-alloc entry when a copy of B would not fit its scratch array.
#include "g950_common.h"

#include <type_traits>
#include <utility>

namespace g950 {

enum GemmMode : int { GEMM_BF16 = 0, GEMM_F16 = 1, GEMM_I8 = 2, GEMM_F32 = 3 };

// MFMAs per 16-byte operand chunk: the 16-bit and int8 forms consume a whole
// chunk per lane in one v_mfma (K 16 / 32); fp32 (v_mfma_f32_32x32x2_f32,
// one value per lane) takes the chunk's four values in four MFMAs
constexpr int mfma_per_chunk(int mode) { return mode == GEMM_F32 ? 4 : 1; }

// 1: whole-slab 16-bit / int8 GEMMs with M, N >= 256 run on 16x16 output
// fragments (gemm_mfma16_body); 0: every shape on the 32x32 form
#ifndef G950_GEMM16
#define G950_GEMM16 1
#endif
constexpr int BM = 256, BN = 256;  // workgroup tile
constexpr int SLAB = 128;          // bytes of K per row per LDS stage (two stages)

// 128 zero bytes: the DMA source of every 16-byte chunk past K in the last
// (partial) K slab, so the tail multiplies zeros instead of reading past a
// row (K % 64 != 0 kernels only)
__device__ __attribute__((aligned(128))) const uint32_t g950_zero_line[32] = {};

// One 16-byte-per-lane global->LDS DMA instruction (global_load_lds_dwordx4,
// scalar base + 32-bit lane offset, LDS destination in M0) written as inline
// asm: the compiler then sees no LDS write in flight and adds no vmcnt wait
// before the transposing LDS reads (ds_read_tr16_b64), whose address it
// cannot compare with a DMA destination.  Completion is the slab protocol's
// explicit vmcnt(0) + barrier.  (s_nop 0: one wait state between the M0
// write and the DMA.)
__device__ __forceinline__ void dma16_asm(const char* sbase, uint32_t voff, uint32_t lds_dst) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds_dst);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(sbase), "{m0}"(m0) : "memory");
}
// the same from a 64-bit lane offset (rows too far apart for 32 bits)
__device__ __forceinline__ void dma16_asm(const char* sbase, long long voff, uint32_t lds_dst) {
  const uint32_t m0 = __builtin_amdgcn_readfirstlane(lds_dst);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(sbase + voff), "{m0}"(m0) : "memory");
}
template <bool FAR>
using DmaOff = std::conditional_t<FAR, long long, uint32_t>;

// Map the linear workgroup id to a (tile_m, tile_n): XCD-contiguous, then
// grouped by 4 tile-rows.  The hardware deals workgroups round-robin over
// the 8 XCDs, so XCD x runs ids x, x + 8, ...: it takes the contiguous run of
// floor(total / 8) tiles (one more for x < total % 8) starting at
// x * floor(total / 8) + min(x, total % 8).  Tile counts that are not a
// multiple of 8 took ids in plain order before: 4097x11008x4096 (731 tiles)
// 283 -> 268 us, the same bits.
__device__ __forceinline__ void tile_of(int pid, int tiles_m, int tiles_n, int& tm, int& tn) {
  const int total = tiles_m * tiles_n;
  const int x = pid & 7;
  pid = x * (total >> 3) + min(x, total & 7) + (pid >> 3);
  const int group = 4;
  const int per_group = group * tiles_n;
  const int gid = pid / per_group;
  const int first = gid * group;
  const int gsize = min(tiles_m - first, group);
  const int in = pid - gid * per_group;
  tm = first + in % gsize;
  tn = in / gsize;
}

// Epilogue: lane holds C[m][n..n+3] for m = row r of each 32-row fragment,
// n = 8q + 4g + {0..3} of each 32-column fragment; (wm0, wn0) is the first
// output row / column of the wave's tile.  UMASK (int8 only): bit 0 A
// unsigned, bit 1 B unsigned -- the accumulator of the offset operands gets
// its exact correction (modulo 2^32, GemmArgs::rsum / csum).
template <int MODE, int FM, int FN, int UMASK = 0, int RF = 32, class FA = f32x16, class IA = i32x16>
__device__ __forceinline__ void gemm_epilogue(const GemmArgs& p, const FA (&accf)[FM][FN],
                                              const IA (&acci)[FM][FN], int wm0, int wn0,
                                              int lane, int m_lo = 0, int n_lo = 0) {
  // only rows >= m_lo and columns >= n_lo are stored (a tile computed over a
  // window shifted back from the matrix edge owns only its own part)
  // RF x RF output fragments: lane holds C[m][n..n+3] for m = row lane % RF of
  // each fragment and n = 4 * (lane / RF) + (64 / RF) * 4 * q, q < QN
  constexpr int QN = RF * RF / 256;
  const int r = lane % RF, g = lane / RF;
  const bool vec_ok = ((p.c_s0 & 3) == 0);
  // per-row factors
  bool live[FM];
  float rs[FM];
  uint32_t rcorr[FM];
#pragma unroll
  for (int mi = 0; mi < FM; ++mi) {
    const int m = wm0 + mi * RF + r;
    live[mi] = m < p.M && m >= m_lo;
    rs[mi] = 1.0f;
    rcorr[mi] = 0;
    if constexpr (MODE == GEMM_I8) {
      if (live[mi] && p.sa) rs[mi] = p.sa[m];
      if constexpr (UMASK & 2) rcorr[mi] = live[mi] ? 128u * (uint32_t)p.rsum[m] : 0u;
      if constexpr (UMASK == 3) rcorr[mi] -= 16384u * (uint32_t)p.K;
    }
  }
  // one group: C[m][n..n+3] of fragment (mi, ni), column factors colf
  // (sb for int8, cscale for the 16-bit / fp32 GEMMs) and colc (128 * csum)
  auto group = [&](int mi, int ni, int q, int n, bool full, const float (&colf)[4], const uint32_t (&colc)[4]) {
    const int m = wm0 + mi * RF + r;
    float v[4];
    if constexpr (MODE == GEMM_I8) {
      int iv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) iv[e] = (int)((uint32_t)acci[mi][ni][q * 4 + e] + rcorr[mi] + colc[e]);
      if (p.acc_out) {
        int* dst = p.acc_out + (long long)m * p.acc_s0 + n;
        if (((p.acc_s0 & 3) == 0) && full) {
          *(i32x4*)dst = (i32x4){iv[0], iv[1], iv[2], iv[3]};
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (n + e < p.N && n + e >= n_lo) dst[e] = iv[e];
        }
      }
      if (!p.sa) return;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = ((float)iv[e] * rs[mi]) * colf[e];
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = accf[mi][ni][q * 4 + e];
      if (p.cscale) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] *= colf[e];
      }
    }
    char* crow = (char*)p.c + (long long)m * p.c_s0 * (p.c_dtype == DT_F32 ? 4 : 2);
    if (p.c_dtype == DT_F32) {
      float* dst = (float*)crow + n;
      if (vec_ok && full) {
        *(f32x4*)dst = (f32x4){v[0], v[1], v[2], v[3]};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < p.N && n + e >= n_lo) dst[e] = v[e];
      }
    } else {
      uint16_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = (p.c_dtype == DT_BF16) ? f32_to_bf16(v[e]) : f32_to_f16(v[e]);
      uint16_t* dst = (uint16_t*)crow + n;
      if (vec_ok && full) {
        *(u32x2*)dst = (u32x2){(uint32_t)h[0] | ((uint32_t)h[1] << 16),
                               (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (n + e < p.N && n + e >= n_lo) dst[e] = h[e];
      }
    }
  };
  const bool colwise = MODE == GEMM_I8 || p.cscale;
  if (!colwise) {
    // no column factors: row by row, the stores of a row back to back
    const float one[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    const uint32_t zero[4] = {0u, 0u, 0u, 0u};
#pragma unroll
    for (int mi = 0; mi < FM; ++mi) {
      if (!live[mi]) continue;
#pragma unroll
      for (int ni = 0; ni < FN; ++ni)
#pragma unroll
        for (int q = 0; q < QN; ++q) {
          const int n = wn0 + ni * RF + q * (256 / RF) + g * 4;
          if (n + 3 < n_lo) continue;
          group(mi, ni, q, n, n + 3 < p.N && n >= n_lo && (n & 3) == 0, one, zero);
        }
    }
    return;
  }
  // column factors: loaded once per group of four columns and shared by the
  // fragment rows, as one vector load where the group lies inside N and the
  // vector is aligned -- a scalar load per element cost a load-path slot
  // each (128 per lane per tile for the int8 dequant scale)
  const bool sb_vec = MODE == GEMM_I8 && p.sb && ((uintptr_t)p.sb & 15) == 0;
  const bool cs_vec = MODE != GEMM_I8 && p.cscale &&
                      ((uintptr_t)p.cscale & (p.cscale_dtype == DT_F32 ? 15 : 7)) == 0;
  const bool csum_vec = (UMASK & 1) && ((uintptr_t)p.csum & 15) == 0;
#pragma unroll
  for (int ni = 0; ni < FN; ++ni) {
#pragma unroll
    for (int q = 0; q < QN; ++q) {
      const int n = wn0 + ni * RF + q * (256 / RF) + g * 4;
      if (n >= p.N || n + 3 < n_lo) continue;
      const bool full = n + 3 < p.N && n >= n_lo && (n & 3) == 0;
      float colf[4] = {1.0f, 1.0f, 1.0f, 1.0f};
      uint32_t colc[4] = {0u, 0u, 0u, 0u};
      if constexpr (MODE == GEMM_I8) {
        if (p.sa) {
          if (sb_vec && full) {
            const f32x4 t = *(const f32x4*)(p.sb + n);
#pragma unroll
            for (int e = 0; e < 4; ++e) colf[e] = t[e];
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) colf[e] = (n + e < p.N) ? p.sb[n + e] : 0.0f;
          }
        }
        if constexpr (UMASK & 1) {
          if (csum_vec && full) {
            const i32x4 t = *(const i32x4*)(p.csum + n);
#pragma unroll
            for (int e = 0; e < 4; ++e) colc[e] = 128u * (uint32_t)t[e];
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) colc[e] = (n + e < p.N) ? 128u * (uint32_t)p.csum[n + e] : 0u;
          }
        }
      } else {
        if (cs_vec && full) {
          if (p.cscale_dtype == DT_F32) {
            const f32x4 t = *(const f32x4*)((const float*)p.cscale + n);
#pragma unroll
            for (int e = 0; e < 4; ++e) colf[e] = t[e];
          } else {
            const u32x2 t = *(const u32x2*)((const uint16_t*)p.cscale + n);
            const bool bf = p.cscale_dtype == DT_BF16;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint16_t hb = (uint16_t)(t[e >> 1] >> (16 * (e & 1)));
              colf[e] = bf ? bf16_to_f32(hb) : f16_to_f32(hb);
            }
          }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e)
            colf[e] = (n + e < p.N) ? load_as_f32(p.cscale, n + e, p.cscale_dtype) : 0.0f;
        }
      }
#pragma unroll
      for (int mi = 0; mi < FM; ++mi)
        if (live[mi]) group(mi, ni, q, n, full, colf, colc);
    }
  }
}

// One operand chunk into the accumulator.  fp32: lane half h of both
// operands holds k = 4c + e (c the chunk index of the half), so MFMA e sums
// A[m][k] B[k][n] over the two halves' k -- every k of the slab exactly once,
// in an order both operands share.
template <int MODE>
__device__ __forceinline__ void mfma_step(const u32x4& bfrag, const u32x4& afrag, f32x16& accf,
                                          i32x16& acci) {
  if constexpr (MODE == GEMM_F32) {
    // bit-cast the whole vectors, then index: this compiler reads element 0
    // for every __builtin_bit_cast of a single ext_vector element
    const f32x4 bv = __builtin_bit_cast(f32x4, bfrag), av = __builtin_bit_cast(f32x4, afrag);
#pragma unroll
    for (int e = 0; e < 4; ++e) accf = __builtin_amdgcn_mfma_f32_32x32x2f32(bv[e], av[e], accf, 0, 0, 0);
  } else if constexpr (MODE == GEMM_BF16) {
    accf = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, bfrag),
                                                   __builtin_bit_cast(bf16x8, afrag), accf, 0, 0, 0);
  } else if constexpr (MODE == GEMM_F16) {
    accf = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, bfrag),
                                                  __builtin_bit_cast(f16x8, afrag), accf, 0, 0, 0);
  } else {
    acci = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, bfrag),
                                                 __builtin_bit_cast(i32x4, afrag), acci, 0, 0, 0);
  }
}

// The same for 16x16 fragments: lane (g4, l16) holds 16-byte chunk g4 of row
// l16 of both operands; fp32 takes the chunk's four k in four MFMAs.
template <int MODE>
__device__ __forceinline__ void mfma16_step(const u32x4& bfrag, const u32x4& afrag, f32x4& accf, i32x4& acci) {
  if constexpr (MODE == GEMM_F32) {
    const f32x4 bv = __builtin_bit_cast(f32x4, bfrag), av = __builtin_bit_cast(f32x4, afrag);
#pragma unroll
    for (int e = 0; e < 4; ++e) accf = __builtin_amdgcn_mfma_f32_16x16x4f32(bv[e], av[e], accf, 0, 0, 0);
  } else if constexpr (MODE == GEMM_BF16) {
    accf = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, bfrag),
                                                   __builtin_bit_cast(bf16x8, afrag), accf, 0, 0, 0);
  } else if constexpr (MODE == GEMM_F16) {
    accf = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, bfrag), __builtin_bit_cast(f16x8, afrag),
                                                  accf, 0, 0, 0);
  } else {
    acci = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, bfrag), __builtin_bit_cast(i32x4, afrag),
                                                 acci, 0, 0, 0);
  }
}

// Epilogue of the 16x16 form for a 16-bit output whose tile owns all of its
// window's columns: the wave's 64 x 128 output tile passes through its own
// 16 KiB of LDS and leaves as whole 256-byte row pieces, 16 bytes per lane,
// in non-temporal stores.  Lane (g4, l16) of fragment (mi, ni) holds C[row
// mi*16 + l16][cols ni*16 + 4 g4 .. + 3]: 8 bytes into 16-byte chunk
// ni*2 + g4/2 of its LDS row, the chunk index XOR-swizzled by row & 15 (the
// 16 rows of one write spread over the 64 banks; a read of 16 chunks of one
// row covers them once).  Rows below m_lo belong to the tile above (a
// window shifted back from the bottom edge) and are not stored.  Measured
// on MI355X against row-by-row 8-byte stores: 8192^3 bf16 757 -> 694 us,
// row-major B 785 -> 708, W8A16 8192^3 816 -> 750, int8 4096x8192x8192
// 199 -> 194, 4097x11008x4096 287 -> 281, the same bits; non-temporal 8-byte
// stores without the staging cost 4097x11008x4096 9% and the int8 GEMM 19%
// (partial lines), and the staging with write-back stores gained 1%.
template <int MODE, int FM, int FN, int UMASK>
__device__ __forceinline__ void gemm_epilogue_lds(const GemmArgs& p, const f32x4 (&accf)[FM][FN],
                                                  const i32x4 (&acci)[FM][FN], int wm0, int wn0, int lane,
                                                  int m_lo, char* reg) {
  constexpr int RB = FN * 32;         // bytes of one wave-tile row
  constexpr int CPR = RB / 16;        // 16-byte chunks per row
  constexpr int RPI = 64 / CPR;       // rows per store instruction
  static_assert(CPR == 16, "the row swizzle spans 16 chunks");
  const int l16 = lane & 15, g4 = lane >> 4;
  const bool bf = p.c_dtype == DT_BF16;
  float rs[FM];
  uint32_t rcorr[FM];
#pragma unroll
  for (int mi = 0; mi < FM; ++mi) {
    const int m = wm0 + mi * 16 + l16;
    rs[mi] = 1.0f;
    rcorr[mi] = 0;
    if constexpr (MODE == GEMM_I8) {
      rs[mi] = p.sa[m];
      if constexpr (UMASK & 2) rcorr[mi] = 128u * (uint32_t)p.rsum[m];
      if constexpr (UMASK == 3) rcorr[mi] -= 16384u * (uint32_t)p.K;
    }
  }
#pragma unroll
  for (int ni = 0; ni < FN; ++ni) {
    const int n = wn0 + ni * 16 + g4 * 4;
    float colf[4] = {1.0f, 1.0f, 1.0f, 1.0f};
    uint32_t colc[4] = {0u, 0u, 0u, 0u};
    if constexpr (MODE == GEMM_I8) {
      if (((uintptr_t)p.sb & 15) == 0) {
        const f32x4 t = *(const f32x4*)(p.sb + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) colf[e] = t[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) colf[e] = p.sb[n + e];
      }
      if constexpr (UMASK & 1) {
        if (((uintptr_t)p.csum & 15) == 0) {
          const i32x4 t = *(const i32x4*)(p.csum + n);
#pragma unroll
          for (int e = 0; e < 4; ++e) colc[e] = 128u * (uint32_t)t[e];
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) colc[e] = 128u * (uint32_t)p.csum[n + e];
        }
      }
    } else if (p.cscale) {
      if (p.cscale_dtype == DT_F32 && ((uintptr_t)p.cscale & 15) == 0) {
        const f32x4 t = *(const f32x4*)((const float*)p.cscale + n);
#pragma unroll
        for (int e = 0; e < 4; ++e) colf[e] = t[e];
      } else if (p.cscale_dtype != DT_F32 && ((uintptr_t)p.cscale & 7) == 0) {
        const u32x2 t = *(const u32x2*)((const uint16_t*)p.cscale + n);
        const bool cbf = p.cscale_dtype == DT_BF16;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const uint16_t hb = (uint16_t)(t[e >> 1] >> (16 * (e & 1)));
          colf[e] = cbf ? bf16_to_f32(hb) : f16_to_f32(hb);
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) colf[e] = load_as_f32(p.cscale, n + e, p.cscale_dtype);
      }
    }
#pragma unroll
    for (int mi = 0; mi < FM; ++mi) {
      // the same arithmetic, in the same order, as gemm_epilogue
      float v[4];
      if constexpr (MODE == GEMM_I8) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          v[e] = ((float)(int)((uint32_t)acci[mi][ni][e] + rcorr[mi] + colc[e]) * rs[mi]) * colf[e];
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = accf[mi][ni][e] * colf[e];
      }
      uint16_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = bf ? f32_to_bf16(v[e]) : f32_to_f16(v[e]);
      const int row = mi * 16 + l16, chunk = ni * 2 + (g4 >> 1);
      *(u32x2*)(reg + row * RB + ((chunk ^ l16) << 4) + (g4 & 1) * 8) =
          (u32x2){(uint32_t)h[0] | ((uint32_t)h[1] << 16), (uint32_t)h[2] | ((uint32_t)h[3] << 16)};
    }
  }
  const long long cs = (long long)p.c_s0 * 2;
  char* cbase = (char*)p.c + (long long)wm0 * cs + (long long)wn0 * 2;
#pragma unroll
  for (int it = 0; it < FM * 16 / RPI; ++it) {
    const int r = it * RPI + lane / CPR, c = lane % CPR;
    const u32x4 v = *(const u32x4*)(reg + r * RB + ((c ^ (r & 15)) << 4));
    if (wm0 + r >= m_lo) __builtin_nontemporal_store(v, (u32x4*)(cbase + r * cs + c * 16));
  }
}

// 16x16-fragment form of the 256x256 kernel, for M and N of at least one
// tile: a tile at the bottom / right edge computes the 256 x 256 window
// ending at the matrix edge (every DMA row lies inside the operands, so a
// lane's DMA source is a fixed 32-bit offset plus a wave-uniform base, no
// per-row clamp) and stores only its own rows and columns.
//
// BROW (16-bit only): B is the reference matmul's own row-major [K, N]
// (N-contiguous, ops/suite/perf/matmul.py:33) and is read as it lies, with
// no transposed copy.  A slab's 64 k-rows of the tile's 256 columns land in
// LDS as four 64-column blocks of 64 rows x 128 bytes -- the same 8-row x
// 128-byte DMA instruction as the K-contiguous operands, whole 128-byte
// lines of B -- and each B fragment (16 columns x 8 k per lane) comes out of
// two ds_read_b64_tr_b16 (gfx950's transposing read: in each 16-lane group,
// lane 4r + j reads 4 columns of k-row r and lane i receives column i of the
// four rows).  The 16-byte chunks of k-row k are XOR-swizzled by
// 2 * (((k >> 1) & 1) | (((k >> 3) & 1) << 1)), so the eight k-rows a half
// wave reads (k, k+1, k+2, k+3 and the same eight rows on) cover the 64 banks
// once.  Stages sit as [A0][B0][B1][A1] so a B read of either stage is one
// per-lane base plus an immediate below 64 KiB.
template <int MODE, int WM, int WN, int UMASK, bool BROW = false>
__device__ __forceinline__ void gemm_mfma16_body(const GemmArgs& p, char* lds) {
  constexpr int NW = WM * WN;
  constexpr int STAGE = (BM + BN) * SLAB;     // 64 KiB
  constexpr int DW = NW / 2;                  // DMA waves: the first half, one per SIMD
  constexpr int GROUPS = (BM + BN) / 8 / DW;  // 8-row DMA groups per DMA wave per slab
  constexpr int H = GROUPS / 2;
  static_assert(GROUPS * 8 * DW == BM + BN && GROUPS % 2 == 0 && (BM / 8) % GROUPS == 0,
                "each DMA wave's groups lie in one operand");
  static_assert(!BROW || (MODE == GEMM_BF16 || MODE == GEMM_F16), "row-major B: 16-bit operands");
  // LDS byte offsets of stage s's A and B slabs
  constexpr int A_OFF[2] = {0, BROW ? STAGE + BN * SLAB : STAGE};
  constexpr int B_OFF[2] = {BM * SLAB, BROW ? BM * SLAB + BN * SLAB : STAGE + BM * SLAB};
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN;
  const int wn = wave % WN;
  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
  const int m_own = tm * BM, n_own = tn * BN;
  const int m0 = min(m_own, p.M - BM);  // the window the tile computes
  const int n0 = min(n_own, p.N - BN);
  constexpr int ES = (MODE == GEMM_I8) ? 1 : 2;  // element bytes
  const long long lda_b = p.a_s0 * ES;
  const long long ldb_b = p.b_s0 * ES;
  const char* abase = (const char*)p.a + (long long)m0 * lda_b;
  const char* bbase = (const char*)p.b + (long long)n0 * ldb_b;
  const int kslabs = p.K * ES / SLAB;
  const int last = kslabs - 1;
  // DMA: wave w < DW owns row groups w*GROUPS .. +GROUPS-1 (A rows for the
  // first BM/8 groups, B rows after), 8 rows x 128 bytes per instruction
  // (lane: row lane / 8, 16-byte slot lane % 8 holding chunk slot ^ ((row >>
  // 1) & 7)).  Group t's rows are the first group's plus 8t, and the
  // swizzle repeats every second group, so a lane needs two offsets.
  // Row-major B: group g (of the slab's 32) is column block g / 8, k-rows
  // 8 (g % 8) .. +7; its swizzle repeats every second group too.
  const bool dma_a = wave * GROUPS < BM / 8;
  const bool dma_brow = BROW && !dma_a;
  const long long ld = dma_a ? lda_b : ldb_b;
  // per-slab step of the DMA source: 128 bytes of K, or 64 k-rows of row-major B
  const long long slab_step = dma_brow ? 64 * ldb_b : SLAB;
  const int g0 = dma_a ? wave * GROUPS : wave * GROUPS - BM / 8;  // first group of this wave in its operand
  const char* obase = dma_a ? abase : dma_brow ? (const char*)p.b + (long long)n0 * 2 + (g0 >> 3) * 128 : bbase;
  uint32_t doff[2];
  {
    const int r8 = lane >> 3;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if (dma_brow) {
        const int k = 8 * j + r8;
        const int sw = 2 * (((k >> 1) & 1) | (((k >> 3) & 1) << 1));
        doff[j] = (uint32_t)((long long)k * ld + (((lane & 7) ^ sw) * 16));
      } else {
        const int row = g0 * 8 + r8 + 8 * j;
        doff[j] = (uint32_t)((long long)row * ld + (((lane & 7) ^ ((row >> 1) & 7)) * 16));
      }
    }
  }
  // LDS byte address of the stages (the asm DMA's M0)
  const uint32_t lds32 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)lds;
  auto issue = [&](int stage, int slab, int t0, int t1) {
    char* st = lds + (dma_a ? A_OFF[stage] : B_OFF[stage]);
#pragma unroll
    for (int t = t0; t < t1; ++t) {
      // wave-uniform part of group t's source: column block and row pair
      const long long grp = dma_brow ? (long long)(t >> 3) * 128 + (long long)((t & 7) & ~1) * 8 * ld
                                     : (long long)(t & ~1) * 8 * ld;
      const char* ub = obase + (long long)slab * slab_step + grp;
      if constexpr (BROW) {
        dma16_asm(ub, doff[t & 1], lds32 + (uint32_t)((dma_a ? A_OFF[stage] : B_OFF[stage]) + (g0 + t) * 1024));
      } else {
        asm volatile("" : "+v"(doff[t & 1]));
        const char* src = ub + (uint64_t)doff[t & 1];
        __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                         (__attribute__((address_space(3))) void*)(st + (g0 + t) * 1024),
                                         16, 0, 0);
      }
    }
  };
  // ---- 16x16 output fragments (v_mfma_f32_16x16x32_{bf16,f16} /
  // v_mfma_i32_16x16x64_i8: 16 bytes of K per lane, the 64-byte k-step
  // split over the four 16-lane groups).  Under the power limit these
  // sustain more FLOP/s than the 32x32x16 form with the same operand
  // traffic (half the accumulator register traffic per FLOP).  Wave tile
  // 64 x 128 = 4 x 8 fragments; per slab two k-steps of 64 bytes.  Lane
  // (g4, l16) reads row l16 of each 16-row fragment, chunk 4 ks + g4; the
  // swizzle (row >> 1) & 7 depends on l16 alone, so fragment i is the
  // lane's offset plus an immediate i * 16 rows (conflict-free: each
  // 16-lane group covers the 64 banks once).
  constexpr int FM16 = BM / WM / 16, FN16 = BN / WN / 16;
  f32x4 acf[FM16][FN16];
  i32x4 aci[FM16][FN16];
#pragma unroll
  for (int i = 0; i < FM16; ++i)
#pragma unroll
    for (int j = 0; j < FN16; ++j) {
      if constexpr (MODE == GEMM_I8) aci[i][j] = (i32x4){};
      else acf[i][j] = (f32x4){};
    }
  const int l16 = lane & 15, g4 = lane >> 4;
  int aoff[2][2], boff[2][2];
#pragma unroll
  for (int s_ = 0; s_ < 2; ++s_)
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      const int sw = (((ks * 4 + g4) ^ ((l16 >> 1) & 7)) << 4) + l16 * SLAB;
      aoff[s_][ks] = A_OFF[s_] + wm * (BM / WM) * SLAB + sw;
      boff[s_][ks] = B_OFF[s_] + wn * (BN / WN) * SLAB + sw;
    }
  // Row-major B fragment ni of k-step ks: lane (g4, 4 r + j) reads k-rows
  // 32 ks + 8 g4 + r (and + 4) at columns 4 j .. 4 j + 3 of the fragment's 16,
  // in column block 2 wn + ni / 4, chunk pair (ni % 4) ^ swizzle: the lane's
  // base for each ni % 4 (stage 0), everything else an immediate (stage 1 is
  // the next 32 KiB).
  int btr[4];
  if constexpr (BROW) {
    const int r = l16 >> 2, j = l16 & 3;
    const int sw = ((r >> 1) & 1) | ((g4 & 1) << 1);
#pragma unroll
    for (int cp = 0; cp < 4; ++cp)
      btr[cp] = B_OFF[0] + (2 * wn) * 64 * SLAB + (8 * g4 + r) * SLAB + 32 * (cp ^ sw) + 8 * j;
  }
  u32x4 a16[2][FM16], b16[FN16];
  auto afrag = [&](auto sc, int ks, int buf) {
    constexpr int S = decltype(sc)::value;
#pragma unroll
    for (int mi = 0; mi < FM16; ++mi) a16[buf][mi] = *(const u32x4*)(lds + aoff[S][ks] + mi * 16 * SLAB);
  };
  auto bfrag = [&](auto sc, int ks, int ni) {
    constexpr int S = decltype(sc)::value;
    if constexpr (BROW) {
      typedef short s16x4 __attribute__((ext_vector_type(4)));
      const int off = btr[ni & 3] + S * BN * SLAB + (ni >> 2) * 64 * SLAB + ks * 32 * SLAB;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(lds + off));
      const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
          (__attribute__((address_space(3))) s16x4*)(lds + off + 4 * SLAB));
      const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
      b16[ni] = (u32x4){l2[0], l2[1], h2[0], h2[1]};
    } else {
      b16[ni] = *(const u32x4*)(lds + boff[S][ks] + ni * 16 * SLAB);
    }
  };
  auto mma = [&](const u32x4& bv, const u32x4& av, f32x4& cf, i32x4& ci) {
    if constexpr (MODE == GEMM_BF16)
      cf = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, bv), __builtin_bit_cast(bf16x8, av),
                                                   cf, 0, 0, 0);
    else if constexpr (MODE == GEMM_F16)
      cf = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, bv), __builtin_bit_cast(f16x8, av), cf,
                                                  0, 0, 0);
    else
      ci = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4, bv), __builtin_bit_cast(i32x4, av), ci,
                                                 0, 0, 0);
  };
  // One k-step: the MFMAs of (a16[buf], b16) with the next k-step's
  // fragments read behind them -- stage NS, k-step nks: A into the other
  // buffer (first four slots), each B fragment into its own registers once
  // its last MFMA has issued -- and ndma DMA instructions spread over the
  // slots; an explicit lgkmcnt(0) closes the k-step (the compiler cannot
  // count LDS reads issued behind a DMA).
  // (BROW: the DMA is inline asm, which the scheduling groups cannot place,
  // so the k-step issues its ndma DMA groups itself, dt0.. of slab dslab into
  // stage dst: two among the next k-step's A reads, then one behind each B
  // fragment's reads; the asm keeps its place among the LDS reads.  Issued
  // one behind each B fragment from the first, the last DMA of a k-step
  // lands just before the slab barrier's vmcnt(0): measured 812 -> 798 us at
  // 8192^3.)
  constexpr int NMF16 = FM16 * FN16;
  constexpr int EARLY = 2;  // BROW: DMA groups issued among the A reads
  auto kstep = [&](auto bc, auto nsc, int nks, int ndma, int dst = 0, int dslab = 0, int dt0 = 0) {
    constexpr int buf = decltype(bc)::value;
    if constexpr (BROW) {
      constexpr int S = decltype(nsc)::value;
#pragma unroll
      for (int mi = 0; mi < FM16; ++mi) {
        a16[buf ^ 1][mi] = *(const u32x4*)(lds + aoff[S][nks] + mi * 16 * SLAB);
        if (mi >= 1 && mi <= EARLY && mi - 1 < ndma) issue(dst, dslab, dt0 + mi - 1, dt0 + mi);
      }
    } else {
      afrag(nsc, nks, buf ^ 1);
    }
    if constexpr (UMASK & 1) {
#pragma unroll
      for (int mi = 0; mi < FM16; ++mi) a16[buf][mi] ^= 0x80808080u;
    }
#pragma unroll
    for (int ni = 0; ni < FN16; ++ni) {
      if constexpr (UMASK & 2) b16[ni] ^= 0x80808080u;
#pragma unroll
      for (int mi = 0; mi < FM16; ++mi) mma(b16[ni], a16[buf][mi], acf[mi][ni], aci[mi][ni]);
      bfrag(nsc, nks, ni);
      if constexpr (BROW) {
        const int dj = ni + EARLY;
        if (dj < ndma) issue(dst, dslab, dt0 + dj, dt0 + dj + 1);
      }
    }
#pragma unroll
    for (int i = 0; i < NMF16; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (i < FM16) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (i % FM16 == FM16 - 1) __builtin_amdgcn_sched_group_barrier(0x100, BROW ? 2 : 1, 0);
      if (!BROW && ndma && i % (NMF16 / ndma) == 1 && i / (NMF16 / ndma) < ndma)
        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  };
  // Two-stage protocol as below, with two k-steps per slab: the barrier
  // sits between them, after every read of slab kt (k-step 1's fragments
  // are read during k-step 0) and after the slab kt + 1 DMA landed.
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  const bool dwave = wave < DW;
  if (dwave) issue(0, 0, 0, GROUPS);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  afrag(S0{}, 0, 0);
#pragma unroll
  for (int ni = 0; ni < FN16; ++ni) bfrag(S0{}, 0, ni);
  if (dwave) issue(1, min(1, last), 0, H);
  __builtin_amdgcn_s_waitcnt(0xc07f);
  auto run = [&](auto dc) {
    constexpr bool DMA = decltype(dc)::value;
    auto slab_iter = [&](auto cc, int kt) {
      constexpr int CUR = decltype(cc)::value, NXT = CUR ^ 1;
      if constexpr (DMA && !BROW) issue(NXT, min(kt + 1, last), H, GROUPS);
      kstep(S0{}, cc, 1, DMA ? H : 0, NXT, min(kt + 1, last), H);
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (DMA && !BROW) issue(CUR, min(kt + 2, last), 0, H);
      // (after the last slab: a stale stage, never used)
      kstep(S1{}, std::integral_constant<int, NXT>{}, 0, DMA ? H : 0, CUR, min(kt + 2, last), 0);
    };
    int kt = 0;
    for (; kt + 1 < kslabs; kt += 2) {
      slab_iter(S0{}, kt);
      slab_iter(S1{}, kt + 1);
    }
    if (kt < kslabs) slab_iter(S0{}, kt);
  };
  if (dwave) run(std::true_type{});
  else run(std::false_type{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // 16-bit output, the tile owning its window's columns, 16-byte aligned
  // rows: staged through LDS (uniform over the workgroup, so every wave
  // reaches the barrier that frees the stages: each wave's reads ended with
  // its last k-step's lgkmcnt(0), each DMA wave's loads with the vmcnt(0))
  if (n0 == n_own && p.c_dtype != DT_F32 && (p.c_s0 & 7) == 0 && ((uintptr_t)p.c & 15) == 0 &&
      (MODE != GEMM_I8 || (p.sa && !p.acc_out))) {
    __syncthreads();
    gemm_epilogue_lds<MODE, FM16, FN16, UMASK>(p, acf, aci, m0 + wm * (BM / WM), n0 + wn * (BN / WN), lane, m_own,
                                               lds + wave * (BM / WM) * (BN / WN) * 2);
    return;
  }
  gemm_epilogue<MODE, FM16, FN16, UMASK, 16>(p, acf, aci, m0 + wm * (BM / WM), n0 + wn * (BN / WN), lane, m_own,
                                              n_own);
}

// 16 int8 -> 16 exact 16-bit floats, as two 8-element operands (k 0..7, 8..15)
template <bool F16>
__device__ __forceinline__ void widen_i8x16(const u32x4& w, u32x4& lo, u32x4& hi) {
  uint32_t o[8];
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const int x = (int)w[d];
    const float f0 = (float)((x << 24) >> 24), f1 = (float)((x << 16) >> 24);
    const float f2 = (float)((x << 8) >> 24), f3 = (float)(x >> 24);
    if constexpr (F16) {
      o[2 * d] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){f0, f1}, f16x2));
      o[2 * d + 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){f2, f3}, f16x2));
    } else {
      o[2 * d] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){f0, f1}, bf16x2));
      o[2 * d + 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){f2, f3}, bf16x2));
    }
  }
  lo = (u32x4){o[0], o[1], o[2], o[3]};
  hi = (u32x4){o[4], o[5], o[6], o[7]};
}

constexpr int W8_LDS = 144 * 1024;  // of the tiled int8-weight kernels

// Smaller workgroup tiles of the whole-slab kernels (GemmArgs::tile), for
// shapes whose 256 x 256 tiles would leave most CUs idle: TM x TN outputs,
// 8 waves as 2 x 2 wave tiles x 2 halves of each K slab (a wave multiplies
// one 64-byte k-step of every slab, so its fragments are read once for a
// (TM/2) x (TN/2) tile: half the LDS reads per MFMA of eight smaller wave
// tiles).  The slabs run through a ring of NST stages filled by direct DMA,
// every wave issuing its share: NST - 1 slabs are in flight, since with few
// MFMAs per slab the latency of a load, not its issue, is what a two-stage
// ring would show.  What bounds it is loading 16, 24 or 32 KB per slab: all
// three tiles run at about 70 bytes per ns and CU with about 100 KB in flight,
// which a latency of 1.4 us explains as well as a limit of the path (the two
// were not told apart).  bf16 512 x 4096 x 4096 68 -> 26 us (64 x 128 tiles,
// one per CU), 256 x 4096 x 4096 68 -> 16, 1000 x 4096 x 4096 68 -> 39,
// int8 512 x 8192 x 8192 70 -> 40, fp32 512 x 2048 x 2048 452 -> 40 (operands
// in the MALL).  fp32 sums in two chains: error against 64 bits at 512 x 2048
// x 4096 1.14e-6 -> 8.1e-7.  Iteration kt multiplies slab kt from registers while slab
// kt + 1's fragments are read; one barrier per slab, after this wave's loads
// of slab kt + 1 have landed.  After it nobody reads slab kt's stage again,
// so slab kt + NST goes there.  The two k-halves of a wave tile are added
// through LDS, each wave finishing half of the rows.
//
// W8 (int8 weights under 16-bit A): a slab is 128 k -- 256 bytes of an A row,
// 128 of a B row -- and a lane's 16 weights are widened as they leave LDS,
// for two MFMAs; B then costs half the bytes.  K need only be a
// multiple of 16: the last slab's chunks past K repeat the row's last one and
// are zeroed in registers.  The column scale is the epilogue's.  It is bound
// by its loads like the others: 512 x 4096 x 4096 30 us, 256 x 4096 x
// 4096 22 and 1024 x 8192 x 8192 153, against 102, 102 and 186 for the 128 x
// 128 kernel it replaced (operands staged through registers, one slab ahead).
//
// BROW (16-bit): row-major B read as it lies (gemm_mfma16_body's notes): a
// slab is 64 k-rows of TN columns, in blocks of 64 columns x 128 bytes, and a
// fragment comes out of two transposing reads; a tile at the right edge
// computes the TN columns ending there and stores its own.  bf16 512 x 4096 x
// 4096 97.6 -> 34 us, 300 x 2048 x 2048 41.8 -> 11.7, 1024 x 8192 x 8192 183 ->
// 152, against the 256 x 256 form; 8192^3 as before.
//
// FAR: 64-bit lane offsets, for rows of A or Bt that lie too far apart (or
// at negative strides) for 32 bits within a tile.
template <int MODE, int TM, int TN, int UMASK, int NST, bool W8 = false, bool BROW = false, bool FAR = false>
__device__ __forceinline__ void gemm_tile_body(const GemmArgs& p, char* lds) {
  constexpr int AROW = W8 ? 256 : SLAB;            // bytes of an A row per slab
  constexpr int STAGE = TM * AROW + TN * SLAB;
  constexpr int AG = TM * AROW / 1024;             // DMA instructions (1 KiB) of A per slab
  constexpr int DPW = STAGE / 8192;                // DMA instructions per wave per slab
  constexpr int AV = W8 ? 2 : 1;                   // A chunks of a lane per fragment
  constexpr int FM = TM / 32, FN = TN / 32;        // 16x16 fragments of a wave tile
  static_assert(NST * STAGE <= (W8 ? W8_LDS : 4 * BM * SLAB) && NST >= 3 && DPW * 8192 == STAGE, "LDS");
  static_assert(FM % 2 == 0 && 8 * (FM / 2) * FN * 1024 <= NST * STAGE, "the k-halves' exchange fits the ring");
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int kg = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
  const int m0 = tm * TM, n0 = BROW ? min(tn * TN, p.N - TN) : tn * TN;
  constexpr int ES = W8 ? 1 : (MODE == GEMM_I8) ? 1 : (MODE == GEMM_F32) ? 4 : 2;  // bytes of a B element
  const long long lda = p.a_s0 * (W8 ? 2 : ES), ldb = p.b_s0 * ES;
  const char* abase = (const char*)p.a + (long long)m0 * lda;
  const char* bbase = (const char*)p.b + (BROW ? (long long)n0 * ES : (long long)n0 * ldb);
  const long long bstep = BROW ? 64 * ldb : SLAB;  // from slab to slab of B
  const int kslabs = (p.K * ES + SLAB - 1) / SLAB;
  const int tb = p.K * ES - (kslabs - 1) * SLAB;   // bytes of the last slab
  // group t of this wave: 8 rows of A or B (rows past the edge repeat the
  // last one; their outputs are not stored), the 16-byte chunks XOR-swizzled
  // by (row >> 1) & 7 as in the 256 x 256 kernels
  DmaOff<FAR> doff[DPW];
  const uint32_t lds32 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)lds;
  // this lane's 16-byte chunk of DMA instruction grp
  auto chunk = [&](int grp) {
    if (W8 && grp < AG) return (lane & 15) ^ ((grp * 4 + (lane >> 4)) & 15);
    if (BROW && grp >= AG) {  // k-row 8 (grp % 8) + lane / 8 of column block (grp - AG) / 8
      const int k = ((grp - AG) & 7) * 8 + (lane >> 3);
      return (lane & 7) ^ (2 * (((k >> 1) & 1) | (((k >> 3) & 1) << 1)));
    }
    const int row = (grp < AG ? grp : grp - AG) * 8 + (lane >> 3);
    return (lane & 7) ^ ((row >> 1) & 7);
  };
#pragma unroll
  for (int t = 0; t < DPW; ++t) {
    const int grp = wave * DPW + t;
    const bool is_a = grp < AG;
    const int row = W8 && is_a ? grp * 4 + (lane >> 4) : (is_a ? grp : grp - AG) * 8 + (lane >> 3);
    if (BROW && !is_a) {
      doff[t] = (uint32_t)((long long)(((grp - AG) & 7) * 8 + (lane >> 3)) * ldb) + ((grp - AG) >> 3) * 128 +
                (chunk(grp) << 4);
      continue;
    }
    const int src = min(row, (is_a ? p.M - m0 : p.N - n0) - 1);
    doff[t] = (DmaOff<FAR>)((long long)src * (is_a ? lda : ldb) + (chunk(grp) << 4));
  }
  auto issue = [&](int slab) {
    const uint32_t dst = lds32 + (uint32_t)(slab % NST) * STAGE;
    const bool tail = W8 && slab == kslabs - 1 && tb != SLAB;
#pragma unroll
    for (int t = 0; t < DPW; ++t) {
      const int grp = wave * DPW + t;
      const bool is_a = grp < AG;
      DmaOff<FAR> off = doff[t];
      if (tail) off -= max(0, (chunk(grp) << 4) + 16 - (is_a ? 2 * tb : tb));
      dma16_asm((is_a ? abase : bbase) + (long long)slab * (is_a ? AROW : bstep), off, dst + grp * 1024);
    }
  };
  const int l16 = lane & 15, g4 = lane >> 4;
  const int kc = kg * 4 + g4;  // this lane's 16-byte chunk of a B row's slab
  const int sw = l16 * SLAB + ((kc ^ ((l16 >> 1) & 7)) << 4);
  const int boff = TM * AROW + wn * (TN / 2) * SLAB + sw;
  int aoff[AV];
  if constexpr (W8) {
#pragma unroll
    for (int q = 0; q < 2; ++q) aoff[q] = (wm * (TM / 2) + l16) * AROW + (((2 * kc + q) ^ l16) << 4);
  } else {
    aoff[0] = wm * (TM / 2) * SLAB + sw;
  }
  // BROW: fragment j is column group cg = wn FN + j of the tile; lane (g4,
  // 4 r + i) reads k-rows 32 kg + 8 g4 + r (and + 4), columns 4 i .. + 3
  int btr[FN];
  if constexpr (BROW) {
    const int r = l16 >> 2;
    const int bsw = ((r >> 1) & 1) | ((g4 & 1) << 1);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int cg = wn * FN + j;
      btr[j] = TM * AROW + (cg >> 2) * 64 * SLAB + (32 * kg + 8 * g4 + r) * SLAB + 32 * ((cg & 3) ^ bsw) + 8 * (l16 & 3);
    }
  }
  u32x4 af[2][FM][AV], bf[2][FN];
  auto frags = [&](int slab, auto bc) {
    constexpr int B = decltype(bc)::value;
    const char* st = lds + (slab % NST) * STAGE;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int q = 0; q < AV; ++q) af[B][i][q] = *(const u32x4*)(st + aoff[q] + i * 16 * AROW);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (BROW) {
        typedef short s16x4 __attribute__((ext_vector_type(4)));
        const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(st + btr[j]));
        const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
            (__attribute__((address_space(3))) s16x4*)(st + btr[j] + 4 * SLAB));
        const u32x2 l2 = __builtin_bit_cast(u32x2, lo), h2 = __builtin_bit_cast(u32x2, hi);
        bf[B][j] = (u32x4){l2[0], l2[1], h2[0], h2[1]};
      } else {
        bf[B][j] = *(const u32x4*)(st + boff + j * 16 * SLAB);
      }
    }
    if (W8 && slab == kslabs - 1 && kc * 16 >= tb) {  // chunks past K
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int q = 0; q < AV; ++q) af[B][i][q] = (u32x4){0u, 0u, 0u, 0u};
#pragma unroll
      for (int j = 0; j < FN; ++j) bf[B][j] = (u32x4){0u, 0u, 0u, 0u};
    }
  };
  f32x4 acf[FM][FN];
  i32x4 aci[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (MODE == GEMM_I8) aci[i][j] = (i32x4){};
      else acf[i][j] = (f32x4){};
    }
  auto mmas = [&](auto bc) {
    constexpr int B = decltype(bc)::value;
    if constexpr (UMASK & 1) {
#pragma unroll
      for (int i = 0; i < FM; ++i) af[B][i][0] ^= 0x80808080u;
    }
    if constexpr (UMASK & 2) {
#pragma unroll
      for (int j = 0; j < FN; ++j) bf[B][j] ^= 0x80808080u;
    }
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (W8) {
        u32x4 lo, hi;
        widen_i8x16<MODE == GEMM_F16>(bf[B][j], lo, hi);
#pragma unroll
        for (int i = 0; i < FM; ++i) mfma16_step<MODE>(lo, af[B][i][0], acf[i][j], aci[i][j]);
#pragma unroll
        for (int i = 0; i < FM; ++i) mfma16_step<MODE>(hi, af[B][i][1], acf[i][j], aci[i][j]);
      } else {
#pragma unroll
        for (int i = 0; i < FM; ++i) mfma16_step<MODE>(bf[B][j], af[B][i][0], acf[i][j], aci[i][j]);
      }
    }
  };
  using B0 = std::integral_constant<int, 0>;
  using B1 = std::integral_constant<int, 1>;
  // this wave's loads of slab s have landed, at most the NST - 2 later ones
  // still in flight (all of them waited for where fewer were issued)
  auto landed = [&](int s) {
    if (s + NST - 2 < kslabs) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * DPW) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  // first NST - 1 slabs; slab kt + NST - 1 is issued before iteration kt's
  // wait, so that wait leaves NST - 2 slabs in flight
  for (int s = 0; s < NST - 1 && s < kslabs; ++s) issue(s);
  landed(0);
  asm volatile("s_barrier" ::: "memory");
  frags(0, B0{});
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  if (NST - 1 < kslabs) issue(NST - 1);
  auto iter = [&](int kt, auto bc) {
    constexpr int B = decltype(bc)::value;
    if (kt + 1 < kslabs) {
      landed(kt + 1);
      asm volatile("s_barrier" ::: "memory");
      if (kt + NST < kslabs) issue(kt + NST);
      frags(kt + 1, std::integral_constant<int, B ^ 1>{});
    }
    mmas(bc);
    // the fragments read above are in registers before the next barrier
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };
  int kt = 0;
  for (; kt + 1 < kslabs; kt += 2) {
    iter(kt, B0{});
    iter(kt + 1, B1{});
  }
  if (kt < kslabs) iter(kt, B0{});

  // ---- add the two k-halves: each wave keeps half of its rows' fragments
  // and hands the other half to its partner (wave ^ 4)
  constexpr int HM = FM / 2;
  __syncthreads();
  char* mine = lds + wave * HM * FN * 1024 + lane * 16;
#pragma unroll
  for (int i = 0; i < HM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      u32x4 v;
      if constexpr (MODE == GEMM_I8) v = __builtin_bit_cast(u32x4, kg ? aci[i][j] : aci[i + HM][j]);
      else v = __builtin_bit_cast(u32x4, kg ? acf[i][j] : acf[i + HM][j]);
      *(u32x4*)(mine + (i * FN + j) * 1024) = v;
    }
  __syncthreads();
  const char* theirs = lds + (wave ^ 4) * HM * FN * 1024 + lane * 16;
  f32x4 hf[HM][FN];
  i32x4 hi[HM][FN];
#pragma unroll
  for (int i = 0; i < HM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const u32x4 v = *(const u32x4*)(theirs + (i * FN + j) * 1024);
      // k-half 0 first on both waves
      if constexpr (MODE == GEMM_I8) hi[i][j] = (kg ? aci[i + HM][j] : aci[i][j]) + __builtin_bit_cast(i32x4, v);
      else hf[i][j] = (kg ? acf[i + HM][j] : acf[i][j]) + __builtin_bit_cast(f32x4, v);
    }
  gemm_epilogue<MODE, HM, FN, UMASK, 16>(p, hf, hi, m0 + wm * (TM / 2) + kg * HM * 16, n0 + wn * (TN / 2), lane, 0,
                                         tn * TN);
}

// WM x WN waves; wave tile (BM/WM) x (BN/WN) = FM x FN fragments of 32x32.
// UMASK (int8): bit 0 A unsigned, bit 1 B unsigned.  An unsigned operand's
// bytes are flipped (XOR 0x80: u - 128, a signed int8) as its fragments enter
// the MFMA; the epilogue adds the exact correction.
template <int MODE, int WM, int WN, int UMASK = 0, bool KTAIL = false>
__device__ __forceinline__ void gemm_mfma_body(const GemmArgs& p) {
  constexpr int NW = WM * WN;
  constexpr int FM = BM / WM / 32;
  constexpr int FN = BN / WN / 32;
  constexpr int STAGE = (BM + BN) * SLAB;     // 64 KiB
  constexpr int DW = NW / 2;                  // DMA waves: the first half, one per SIMD
  constexpr int GROUPS = (BM + BN) / 8 / DW;  // 8-row DMA groups per DMA wave per slab
  constexpr int H = GROUPS / 2;
  static_assert(GROUPS * 8 * DW == BM + BN && GROUPS % 2 == 0, "DMA split over waves and halves");
  __shared__ __attribute__((aligned(1024))) char lds[2 * STAGE];
  if constexpr (!KTAIL && UMASK == 0) {
    // smaller tiles where 256 x 256 ones would leave CUs idle (uniform per
    // launch; the host's gemm_pick_tile)
    if (p.tile == GEMM_TILE_128x128) {
      gemm_tile_body<MODE, 128, 128, UMASK, 4>(p, lds);
      return;
    }
    if (p.tile == GEMM_TILE_64x128) {
      gemm_tile_body<MODE, 64, 128, UMASK, 5>(p, lds);
      return;
    }
    if (p.tile == GEMM_TILE_64x64) {
      gemm_tile_body<MODE, 64, 64, UMASK, 8>(p, lds);
      return;
    }
  }
  if constexpr (G950_GEMM16 && MODE != GEMM_F32 && !KTAIL) {
    // whole-slab 16-bit / int8 GEMMs of at least one tile each way take the
    // 16x16-fragment form (uniform per launch)
    if (p.M >= BM && p.N >= BN) {
      gemm_mfma16_body<MODE, WM, WN, UMASK>(p, lds);
      return;
    }
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN;
  const int wn = wave % WN;
  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, tm, tn);
  const int m0 = tm * BM;
  const int n0 = tn * BN;
  constexpr int ES = (MODE == GEMM_I8) ? 1 : (MODE == GEMM_F32) ? 4 : 2;  // element bytes
  const long long lda_b = p.a_s0 * ES;
  const long long ldb_b = p.b_s0 * ES;  // Bt row stride (n) in bytes
  const char* abase = (const char*)p.a + (long long)m0 * lda_b;
  const char* bbase = (const char*)p.b + (long long)n0 * ldb_b;
  const int a_lim = p.M - 1 - m0;
  const int b_lim = p.N - 1 - n0;
  // KTAIL: K need only be a whole number of 16-byte chunks; the last slab's
  // chunks past K come from g950_zero_line
  const int kbytes = p.K * ES;
  const int kslabs = KTAIL ? (kbytes + SLAB - 1) / SLAB : kbytes / SLAB;
  const int last = kslabs - 1;

  f32x16 accf[FM][FN];
  i32x16 acci[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      if constexpr (MODE == GEMM_I8) acci[i][j] = (i32x16){};
      else accf[i][j] = (f32x16){};
    }

  // DMA: one wave instruction moves 8 rows x 128 bytes (lane: row lane / 8,
  // 16-byte slot lane % 8, which holds the swizzled chunk).  Row groups
  // 0..BM/8-1 are A rows, the rest B rows; DMA wave w (w < DW) owns groups
  // w*GROUPS .. w*GROUPS+GROUPS-1, issued in two halves.  Waves are dealt to
  // the four SIMDs round-robin, so each SIMD pairs one DMA wave with one
  // wave that only multiplies: while the DMA wave waits on the load path
  // (every wave issuing at once left both waves of a SIMD stalled together),
  // the other keeps the matrix core busy (measured on MI355X at 8192^3:
  // 1361 -> 1415 TFLOP/s).
  const int dr = lane >> 3;
  const int dslot = lane & 7;
  // Whole-slab kernels: a lane's DMA rows are fixed for the whole kernel, so
  // its byte offsets from the operand base are computed once (32-bit: the
  // host routes operands whose rows reach past 4 GiB to the _kt kernels) and
  // each slab's source is a wave-uniform base plus that offset -- the
  // scalar-base form of the load, no vector address arithmetic per DMA.  The
  // empty asm re-defines the offset inside the loop so instruction selection
  // sees the (scalar + 32-bit lane offset) shape there instead of a 64-bit
  // address hoisted out of it.  _kt kernels keep 64-bit addresses.
  uint32_t doff[GROUPS];
#pragma unroll
  for (int t = 0; t < GROUPS; ++t) {
    const int rg = wave * GROUPS + t;
    const bool is_a = rg < BM / 8;
    const int row = (is_a ? rg : rg - BM / 8) * 8 + dr;
    const int grow = min(row, is_a ? a_lim : b_lim);
    const int chunk = dslot ^ ((row >> 1) & 7);
    doff[t] = (uint32_t)((long long)grow * (is_a ? lda_b : ldb_b) + chunk * 16);
  }
  auto issue = [&](int stage, int slab, int t0, int t1) {
    char* st = lds + stage * STAGE;
    const long long kb = (long long)slab * SLAB;
#pragma unroll
    for (int t = t0; t < t1; ++t) {
      const int rg = wave * GROUPS + t;
      const bool is_a = rg < BM / 8;
      const char* src;
      if constexpr (KTAIL) {
        const int row = (is_a ? rg : rg - BM / 8) * 8 + dr;
        const int grow = min(row, is_a ? a_lim : b_lim);
        const int chunk = dslot ^ ((row >> 1) & 7);
        src = (is_a ? abase : bbase) + (long long)grow * (is_a ? lda_b : ldb_b) + kb + chunk * 16;
        if (kb + chunk * 16 >= kbytes) src = (const char*)g950_zero_line;
      } else {
        const char* ub = (is_a ? abase : bbase) + kb;
        asm volatile("" : "+v"(doff[t]));
        src = ub + (uint64_t)doff[t];
      }
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)src,
                                       (__attribute__((address_space(3))) void*)(st + rg * 1024),
                                       16, 0, 0);
    }
  };

  // Fragments of k-step ks (16 bf16 / 32 int8 of K) of one stage: lane
  // (g, r) reads 16 bytes of row r of each 32-row fragment, chunk 2 ks + g.
  const int g = lane >> 5;
  const int r = lane & 31;
  u32x4 af[2][FM], bfr[2][FN];
  // Per-lane LDS offsets of k-step ks's fragments in stage s, computed once:
  // the swizzle (row >> 1) & 7 depends on r alone (fragment rows start at
  // multiples of 32), so fragment mi (ni) is that offset plus an immediate
  // mi (ni) * 32 rows, and the loop does no address arithmetic.
  int aoff[2][4], boff[2][4];
#pragma unroll
  for (int s_ = 0; s_ < 2; ++s_)
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      const int sw = ((((ks * 2 + g) ^ ((r >> 1) & 7))) << 4) + r * SLAB;
      aoff[s_][ks] = s_ * STAGE + wm * (BM / WM) * SLAB + sw;
      boff[s_][ks] = s_ * STAGE + BM * SLAB + wn * (BN / WN) * SLAB + sw;
    }
  auto frags = [&](auto sc, int ks, int buf) {
    constexpr int S = decltype(sc)::value;
#pragma unroll
    for (int mi = 0; mi < FM; ++mi) af[buf][mi] = *(const u32x4*)(lds + aoff[S][ks] + mi * 32 * SLAB);
#pragma unroll
    for (int ni = 0; ni < FN; ++ni) bfr[buf][ni] = *(const u32x4*)(lds + boff[S][ks] + ni * 32 * SLAB);
  };
  auto mfmas = [&](int buf) {
    if constexpr (UMASK & 1) {
#pragma unroll
      for (int mi = 0; mi < FM; ++mi) af[buf][mi] ^= 0x80808080u;
    }
    if constexpr (UMASK & 2) {
#pragma unroll
      for (int ni = 0; ni < FN; ++ni) bfr[buf][ni] ^= 0x80808080u;
    }
#pragma unroll
    for (int mi = 0; mi < FM; ++mi)
#pragma unroll
      for (int ni = 0; ni < FN; ++ni)
        mfma_step<MODE>(bfr[buf][ni], af[buf][mi], accf[mi][ni], acci[mi][ni]);
  };
  // One MFMA per slot; the next k-step's LDS reads in the first FM + FN
  // slots; ndma DMA instructions spread evenly over the slots.  The compiler
  // cannot count LDS reads issued behind a DMA, so each k-step ends with an
  // explicit lgkmcnt(0), by when its reads are long done.
  constexpr int NMF = FM * FN * mfma_per_chunk(MODE);  // MFMAs per k-step
  auto kstep = [&](int buf, int ndma) {
    mfmas(buf);
#pragma unroll
    for (int i = 0; i < NMF; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if (i < FM + FN) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
      if (ndma && i % (NMF / ndma) == 0 && i / (NMF / ndma) < ndma)
        __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0)
  };

  // Two-stage protocol.  Iteration kt consumes slab kt from stage kt % 2.
  // Slab kt + 1 goes to the other stage: its first DMA half in k-step 3 of
  // iteration kt - 1, its second half in k-step 0 of iteration kt, both past
  // the barrier after which nobody reads slab kt - 1 again.  The barrier
  // before k-step 3 comes after every read of slab kt (the k-step 3
  // fragments are read during k-step 2) and after each DMA wave's loads of
  // slab kt + 1 have landed (its vmcnt(0) just before the barrier); k-step 3
  // then reads slab kt + 1's first fragments.
  // Past the end of K the DMA re-reads the last slab into a stage nobody
  // reads again, so the loop body has no branch.
  using S0 = std::integral_constant<int, 0>;
  using S1 = std::integral_constant<int, 1>;
  const bool dwave = wave < DW;
  if (dwave) issue(0, 0, 0, GROUPS);
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
  frags(S0{}, 0, 0);
  if (dwave) issue(1, min(1, last), 0, H);
  __builtin_amdgcn_s_waitcnt(0xc07f);
  // the main loop in two compiled forms, with and without the DMA: same
  // barriers, so the two wave roles stay in step slab by slab; two slabs per
  // trip, so each stage's fragment offsets are compile-time picks (an odd
  // last slab runs from stage 0)
  auto run = [&](auto dc) {
    constexpr bool DMA = decltype(dc)::value;
    auto slab_iter = [&](auto cc, int kt) {
      constexpr int CUR = decltype(cc)::value, NXT = CUR ^ 1;
      if constexpr (DMA) issue(NXT, min(kt + 1, last), H, GROUPS);
      frags(cc, 1, 1);
      kstep(0, DMA ? H : 0);
      frags(cc, 2, 0);
      kstep(1, 0);
      frags(cc, 3, 1);
      kstep(0, 0);
      asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (DMA) issue(CUR, min(kt + 2, last), 0, H);
      frags(std::integral_constant<int, NXT>{}, 0, 0);  // (after the last slab: a stale stage, never used)
      kstep(1, DMA ? H : 0);
    };
    int kt = 0;
    for (; kt + 1 < kslabs; kt += 2) {
      slab_iter(S0{}, kt);
      slab_iter(S1{}, kt + 1);
    }
    if (kt < kslabs) slab_iter(S0{}, kt);
  };
  if (dwave) run(std::true_type{});
  else run(std::false_type{});
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  gemm_epilogue<MODE, FM, FN, UMASK>(p, accf, acci, m0 + wm * (BM / WM), n0 + wn * (BN / WN), lane);
}

// Bt[n][k] = B[k][n] for 16-bit elements: B [K, N] row-major with row stride
// b_s0 elements (16-byte aligned rows, N % 8 == 0), Bt contiguous [N, K] at
// p.c (K % 8 == 0).  64 x 64 tiles through LDS, one 32-bit slot per element
// with a 65-slot row pitch, so the column reads of the transposition and the
// row writes are both conflict-free; 16-byte loads and stores.
__device__ __forceinline__ void transpose16_body(const GemmArgs& p) {
  __shared__ uint32_t t[64][65];
  const int tiles_n = (p.N + 63) / 64;
  const int k0 = (blockIdx.x / tiles_n) * 64, n0 = (blockIdx.x % tiles_n) * 64;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = threadIdx.x + 256 * i, k = c >> 3, n8 = (c & 7) * 8;
    if (k0 + k < p.K && n0 + n8 < p.N) {
      const u32x4 w = *(const u32x4*)((const uint16_t*)p.b + (long long)(k0 + k) * p.b_s0 + n0 + n8);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        t[k][n8 + 2 * e] = w[e] & 0xFFFFu;
        t[k][n8 + 2 * e + 1] = w[e] >> 16;
      }
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int c = threadIdx.x + 256 * i, n = c >> 3, k8 = (c & 7) * 8;
    if (n0 + n < p.N && k0 + k8 < p.K) {
      u32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) w[e] = t[k8 + 2 * e][n] | (t[k8 + 2 * e + 1][n] << 16);
      *(u32x4*)((uint16_t*)p.c + (long long)(n0 + n) * p.K + k0 + k8) = w;
    }
  }
}

// The same for 32-bit elements (N % 4 == 0, K % 4 == 0): 16-byte vectors of 4.
__device__ __forceinline__ void transpose32_body(const GemmArgs& p) {
  __shared__ uint32_t t[64][65];
  const int tiles_n = (p.N + 63) / 64;
  const int k0 = (blockIdx.x / tiles_n) * 64, n0 = (blockIdx.x % tiles_n) * 64;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = threadIdx.x + 256 * i, k = c >> 4, n4 = (c & 15) * 4;
    if (k0 + k < p.K && n0 + n4 < p.N) {
      const u32x4 w = *(const u32x4*)((const uint32_t*)p.b + (long long)(k0 + k) * p.b_s0 + n0 + n4);
#pragma unroll
      for (int e = 0; e < 4; ++e) t[k][n4 + e] = w[e];
    }
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int c = threadIdx.x + 256 * i, n = c >> 4, k4 = (c & 15) * 4;
    if (n0 + n < p.N && k0 + k4 < p.K) {
      const u32x4 w = {t[k4][n], t[k4 + 1][n], t[k4 + 2][n], t[k4 + 3][n]};
      *(u32x4*)((uint32_t*)p.c + (long long)(n0 + n) * p.K + k0 + k4) = w;
    }
  }
}

// The same for bytes (int8 weights, N % 16 == 0, K % 16 == 0, 16-byte aligned
// rows): 64 x 64 byte tiles, one 16-byte load (a k-row's 16 columns) and one
// 16-byte store (an n-row's 16 k) per thread, bytes staged as 32-bit slots
// with a 65-slot pitch.
__device__ __forceinline__ void transpose8_body(const GemmArgs& p) {
  __shared__ uint32_t t[64][65];
  const int tiles_n = (p.N + 63) / 64;
  const int k0 = (blockIdx.x / tiles_n) * 64, n0 = (blockIdx.x % tiles_n) * 64;
  {
    const int k = threadIdx.x >> 2, n16 = (threadIdx.x & 3) * 16;
    if (k0 + k < p.K && n0 + n16 < p.N) {
      const u32x4 w = *(const u32x4*)((const uint8_t*)p.b + (long long)(k0 + k) * p.b_s0 + n0 + n16);
#pragma unroll
      for (int e = 0; e < 16; ++e) t[k][n16 + e] = (w[e >> 2] >> (8 * (e & 3))) & 0xFFu;
    }
  }
  __syncthreads();
  {
    const int n = threadIdx.x >> 2, k16 = (threadIdx.x & 3) * 16;
    if (n0 + n < p.N && k0 + k16 < p.K) {
      u32x4 w = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int e = 0; e < 16; ++e) w[e >> 2] |= t[k16 + e][n] << (8 * (e & 3));
      *(u32x4*)((uint8_t*)p.c + (long long)(n0 + n) * p.K + k0 + k16) = w;
    }
  }
}

// Row sums over k of int8 / uint8 operands (I8SumArgs), modulo 2^32: one wave
// per row, 16-byte loads.  A byte's value is (byte ^ 0x80) - 128 when signed,
// the byte itself when unsigned, so every row sums unsigned bytes of
// byte ^ flip and subtracts 128 K for a signed row.
__device__ __forceinline__ uint32_t byte_sum(uint32_t w) {
  const uint32_t t = (w & 0x00FF00FFu) + ((w >> 8) & 0x00FF00FFu);
  return (t & 0xFFFFu) + (t >> 16);
}

__device__ __forceinline__ void i8_sums_body(const I8SumArgs& p) {
  const int lane = threadIdx.x & 63;
  const long long row = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
  if (row >= (long long)p.a_rows + p.b_rows) return;
  const bool is_a = row < p.a_rows;
  const char* src = is_a ? (const char*)p.a + row * p.a_s0 : (const char*)p.b + (row - p.a_rows) * p.b_s0;
  const bool sgn = is_a ? p.a_signed : p.b_signed;
  const uint32_t flip = sgn ? 0x80808080u : 0u;
  uint32_t s = 0;
  const int full = p.K / 16;
  for (int c = lane; c < full; c += 64) {
    const u32x4 w = __builtin_nontemporal_load((const u32x4*)(src + (long long)c * 16));
    s += byte_sum(w[0] ^ flip) + byte_sum(w[1] ^ flip) + byte_sum(w[2] ^ flip) + byte_sum(w[3] ^ flip);
  }
  for (int k = full * 16 + lane; k < p.K; k += 64) s += (uint32_t)(((const uint8_t*)src)[k] ^ (flip & 0xFFu));
  s = __builtin_bit_cast(uint32_t, wave_reduce<OpSumU32>(__builtin_bit_cast(float, s)));
  if (lane == 0) p.out[row] = (int)(s - (sgn ? 128u * (uint32_t)p.K : 0u));
}

// --------------------------------------------- fused weight dequantisation
// W8A16 (dequantize_matmul fused into the GEMM): Y = A . (B * scale[n]) for A
// bf16/fp16 [M,K] (K-contiguous) and B int8 stored as Bt[N,K] (K-contiguous),
// scale per column (ops/suite/perf/dequantize_matmul.py:28-43 followed by
// matmul.py:21-37).  int8 values are exact in bf16/fp16, so A.B accumulates
// exactly as the unfused pair would from exact weights; the scale multiplies
// the fp32 accumulator and the result rounds once at the store.
template <int MODE, bool FAR = false>
__device__ __forceinline__ void gemm_w8a16_tiles(const GemmArgs& p) {
  __shared__ __attribute__((aligned(1024))) char lds[W8_LDS];
  if (blockDim.x != 512) return;  // launch shape must match the kernel
  if (p.tile == GEMM_TILE_128x128) gemm_tile_body<MODE, 128, 128, 0, 3, true, false, FAR>(p, lds);
  else if (p.tile == GEMM_TILE_64x128) gemm_tile_body<MODE, 64, 128, 0, 4, true, false, FAR>(p, lds);
  else gemm_tile_body<MODE, 64, 64, 0, 6, true, false, FAR>(p, lds);
}

// Exact copy of an int8 weight matrix Bt[N, K] (row stride b_s0 bytes, K a
// multiple of 16) into a contiguous bf16 / f16 Bt[N, K] at p.c: one thread per
// 16 int8 values, one 16-byte load and two 16-byte stores.  Every int8 value
// is representable in both formats, so the copy loses nothing.
template <bool F16>
__device__ __forceinline__ void widen_i8_body(const GemmArgs& p) {
  const long long chunks = p.K / 16;
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)p.N * chunks) return;
  const long long n = i / chunks, c = i - n * chunks;
  const u32x4 w = *(const u32x4*)((const char*)p.b + n * p.b_s0 + c * 16);
  u32x4 lo, hi;
  widen_i8x16<F16>(w, lo, hi);
  u32x4* dst = (u32x4*)((char*)p.c + (n * p.K + c * 16) * 2);
  dst[0] = lo;
  dst[1] = hi;
}

// ------------------------------------------------ few rows of A (decode)
// Y = A . B for M <= 64 rows and K-contiguous operands, in every GEMM mode,
// and with int8 weights (W8: A bf16 / f16, B int8 widened exactly, the column
// scale in the epilogue).  Such a product is bound by reading B once, and a
// tiled kernel would leave it to few CUs.  A workgroup owns 16 T columns and
// all of K; its W waves take 128-byte units of K in turn, each through its own
// LDS ring of NS units filled by direct DMA -- instructions of 8 whole
// 128-byte lines -- and waits for its own loads only, so the loop holds no
// barrier.  B rows feed the MFMA A port and the 16 R rows of A (from L2) the
// B port, in the tiled kernels' LDS layout.  The waves' partial tiles are
// added in wave order through LDS: no workspace, no second launch, the same
// bits every run.  Measured on MI355X with operands from HBM: bf16 16 x 4096
// x 4096 17.3 (64 x 64 tiles) -> 10.0 us, 16 x 11008 x 4096 21.5 -> 18.7, 64
// x 4096 x 4096 22.3 -> 14.8; int8 weights 16 x 8192 x 8192 23.1 (each lane
// loading its own operand chunks, 64-byte pieces of 16 rows) -> 18.8, 16 x
// 11008 x 4096 21.0 -> 12.8, 64 x 8192 x 8192 48.7 -> 29.9.  About 5 us of
// these are the launch and the first loads; the rest is HBM.
// FEW: M <= 8 (W8: 4), one DMA instruction brings all of A's unit; the other
// rows of the operand hold whatever LDS holds and feed outputs that are not
// stored (an output row depends on its own row of A alone).
// FAR: 64-bit lane offsets (gemm_tile_body's notes).
// With int8 weights and FEW each workgroup starts at its own place in K (the
// golden ratio's multiples spread them evenly) and wraps round: where all
// workgroups walk K in step, rows of 8 KiB or so keep them on the same few
// HBM channels.  One row of A, from 0 -> spread (us; the kernel that loaded
// operands into registers, each wave its own part of K): 4096 x 11008 14.4 ->
// 11.4 (13.2), 8192 x 22016 42.8 -> 32.6 (38.2), 16384 x 8192 30.0 -> 25.6
// (26.4), 4096 x 8192 9.7 -> 9.4 (9.1); at K = 14336, 112 whole units, it is
// 3% behind walking in step (16384 columns 42.4 -> 43.7; 45.3).
// A4: the unit holds FEW's four rows of A alone, so that two workgroups fit a
// CU: for grids of more than one round (gemm_w8a16_few).
constexpr int FEW_LDS = 160 * 1024;

template <int MODE, bool W8, int R, int T, int W, int NS, bool FEW = false, bool FAR = false, bool A4 = false>
__device__ __forceinline__ void gemm_stream_body(const GemmArgs& p, char* lds) {
  constexpr int ES = W8 ? 1 : (MODE == GEMM_I8) ? 1 : (MODE == GEMM_F32) ? 4 : 2;  // bytes of a B element
  constexpr int AROW = W8 ? 256 : 128;       // bytes of an A row's unit
  static_assert(!A4 || (W8 && FEW && R == 1), "four rows of A");
  constexpr bool SPREAD = W8 && FEW;
  constexpr int AU = A4 ? 1024 : 16 * R * AROW, BU = 16 * T * 128, UNIT = AU + BU;
  constexpr int DA = FEW ? 1 : AU / 1024, DB = BU / 1024, DPU = DA + DB;
  static_assert(W * NS * UNIT <= FEW_LDS && NS >= 2 && R * T * 1024 <= NS * UNIT, "the rings fit LDS");
  if (blockDim.x != W * 64) return;  // launch shape must match the kernel
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int g4 = lane >> 4, l16 = lane & 15;
  const int n0 = blockIdx.x * 16 * T;
  const long long lda = p.a_s0 * (W8 ? 2 : ES), ldb = p.b_s0 * ES;
  const char* abase = (const char*)p.a;
  const char* bbase = (const char*)p.b + (long long)n0 * ldb;
  const int kb = p.K * ES;                   // bytes of a B row
  const int units = (kb + 127) / 128;
  const int tb = kb - (units - 1) * 128;     // bytes of the last unit (a multiple of 16)
  const int nloc = units > wave ? (units - wave + W - 1) / W : 0;
  char* ring = lds + wave * NS * UNIT;
  const uint32_t ring32 = (uint32_t)(uintptr_t)(const __attribute__((address_space(3))) char*)ring;
  // DMA instruction u: 8 rows x 128 bytes (W8's A: 4 rows x 256 bytes), the
  // 16-byte chunks XOR-swizzled by the row.  Rows past M repeat row M - 1 and
  // columns past N column N - 1: their outputs are never stored.
  DmaOff<FAR> aoff[DA], boff[DB];
  auto achunk = [&](int u) {
    const int row = W8 ? u * 4 + (lane >> 4) : u * 8 + (lane >> 3);
    return W8 ? (lane & 15) ^ (row & 15) : (lane & 7) ^ ((row >> 1) & 7);
  };
  auto bchunk = [&](int u) { return (lane & 7) ^ (((u * 8 + (lane >> 3)) >> 1) & 7); };
#pragma unroll
  for (int u = 0; u < DA; ++u) {
    const int row = W8 ? u * 4 + (lane >> 4) : u * 8 + (lane >> 3);
    aoff[u] = (DmaOff<FAR>)((long long)min(row, p.M - 1) * lda) + (achunk(u) << 4);
  }
#pragma unroll
  for (int u = 0; u < DB; ++u)
    boff[u] = (DmaOff<FAR>)((long long)min(u * 8 + (lane >> 3), p.N - 1 - n0) * ldb) + (bchunk(u) << 4);
  const int start = SPREAD ? (int)(((uint64_t)(blockIdx.x * 2654435769u) * (uint32_t)units) >> 32) : 0;
  auto unit_of = [&](int j) {  // this wave's j-th unit of K
    const int u = start + wave + W * j;
    return SPREAD && u >= units ? u - units : u;
  };
  auto issue = [&](int j, int slot) {
    const int unit = unit_of(j);
    const char* as = abase + (long long)unit * AROW;
    const char* bs = bbase + (long long)unit * 128;
    const uint32_t dst = ring32 + (uint32_t)slot * UNIT;
    if (unit == units - 1 && tb != 128) {
      // chunks past K repeat the row's last one (zeroed as they are used)
#pragma unroll
      for (int u = 0; u < DB; ++u) dma16_asm(bs, boff[u] - max(0, (bchunk(u) << 4) + 16 - tb), dst + AU + u * 1024);
#pragma unroll
      for (int u = 0; u < DA; ++u)
        dma16_asm(as, aoff[u] - max(0, (achunk(u) << 4) + 16 - tb * (W8 ? 2 : 1)), dst + u * 1024);
    } else {
#pragma unroll
      for (int u = 0; u < DB; ++u) dma16_asm(bs, boff[u], dst + AU + u * 1024);
#pragma unroll
      for (int u = 0; u < DA; ++u) dma16_asm(as, aoff[u], dst + u * 1024);
    }
  };
  f32x4 acf[R][T];
  i32x4 aci[R][T];
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if constexpr (MODE == GEMM_I8) aci[r][t] = (i32x4){};
      else acf[r][t] = (f32x4){};
    }
  for (int j = 0; j < NS && j < nloc; ++j) issue(j, j);
  // unit j lies in slot j % NS; no remainder by 3 in the loop (it cost one row
  // of A with int8 weights up to a fifth: 432 x 28672 21.2 -> 17.1 us)
  for (int j = 0, turn = 0; j < nloc; ++j, turn = turn + 1 == NS ? 0 : turn + 1) {
    const int slot = (NS & (NS - 1)) == 0 ? j % NS : turn;
    // unit j has landed once at most the later units' loads are in flight
    if (j + NS <= nloc) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 1) * DPU) : "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const char* st = ring + slot * UNIT;
    const bool tail = unit_of(j) == units - 1 && tb != 128;
    u32x4 av[2][R][W8 ? 2 : 1], bv[2][T];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int c = 4 * h + g4;
#pragma unroll
      for (int t = 0; t < T; ++t) bv[h][t] = *(const u32x4*)(st + AU + (16 * t + l16) * 128 + ((c ^ ((l16 >> 1) & 7)) << 4));
#pragma unroll
      for (int r = 0; r < R; ++r) {
        if constexpr (W8) {
          const int row = A4 ? l16 & 3 : l16;
          av[h][r][0] = *(const u32x4*)(st + (16 * r + row) * 256 + (((2 * c) ^ row) << 4));
          av[h][r][1] = *(const u32x4*)(st + (16 * r + row) * 256 + (((2 * c + 1) ^ row) << 4));
        } else {
          av[h][r][0] = *(const u32x4*)(st + (16 * r + l16) * 128 + ((c ^ ((l16 >> 1) & 7)) << 4));
        }
      }
      if (tail && c * 16 >= tb) {
#pragma unroll
        for (int t = 0; t < T; ++t) bv[h][t] = (u32x4){0u, 0u, 0u, 0u};
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
          for (int q = 0; q < (W8 ? 2 : 1); ++q) av[h][r][q] = (u32x4){0u, 0u, 0u, 0u};
      }
    }
    // the unit's reads have returned before its slot is refilled
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if (j + NS < nloc) issue(j + NS, slot);
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int t = 0; t < T; ++t) {
        if constexpr (W8) {
          u32x4 lo, hi;
          widen_i8x16<MODE == GEMM_F16>(bv[h][t], lo, hi);
#pragma unroll
          for (int r = 0; r < R; ++r) {
            mfma16_step<MODE>(lo, av[h][r][0], acf[r][t], aci[r][t]);
            mfma16_step<MODE>(hi, av[h][r][1], acf[r][t], aci[r][t]);
          }
        } else {
#pragma unroll
          for (int r = 0; r < R; ++r) mfma16_step<MODE>(bv[h][t], av[h][r][0], acf[r][t], aci[r][t]);
        }
      }
  }
  __syncthreads();  // every wave is done with its ring
#pragma unroll
  for (int r = 0; r < R; ++r)
#pragma unroll
    for (int t = 0; t < T; ++t) {
      f32x4 v;
      if constexpr (MODE == GEMM_I8) v = __builtin_bit_cast(f32x4, aci[r][t]);
      else v = acf[r][t];
      *(f32x4*)(lds + ((wave * R * T + r * T + t) * 64 + lane) * 16) = v;
    }
  __syncthreads();
  // fragment f (rows 16 (f / T), columns 16 (f % T)) is wave f % W's: lane
  // (g4, l16) holds row l16, columns 4 g4 .. + 3
  for (int f = wave; f < R * T; f += W) {
    f32x4 sf[1][1];
    i32x4 si[1][1];
    sf[0][0] = *(const f32x4*)(lds + (f * 64 + lane) * 16);
    si[0][0] = __builtin_bit_cast(i32x4, sf[0][0]);
#pragma unroll
    for (int w = 1; w < W; ++w) {
      const f32x4 v = *(const f32x4*)(lds + ((w * R * T + f) * 64 + lane) * 16);
      if constexpr (MODE == GEMM_I8) si[0][0] += __builtin_bit_cast(i32x4, v);
      else sf[0][0] += v;
    }
    gemm_epilogue<MODE, 1, 1, 0, 16>(p, sf, si, 16 * (f / T), n0 + 16 * (f % T), lane);
  }
}

// The forms of one row class (R groups of 16 rows of A): GemmArgs::tile is
// the column groups T per workgroup, picked by the host with the workgroup
// size that form has (g950rt.cpp, kFewRows).
template <int MODE, bool W8, int R>
__device__ __forceinline__ void gemm_few_rows(const GemmArgs& p, char* lds) {
  if constexpr (R == 1) {
    auto forms = [&](auto few) {
      constexpr bool F = decltype(few)::value;
      if (p.tile == 1) gemm_stream_body<MODE, W8, 1, 1, 8, W8 ? 3 : 4, F>(p, lds);
      else if (p.tile == 3) gemm_stream_body<MODE, W8, 1, 3, 8, 2, F>(p, lds);
      else if (p.tile == 4) gemm_stream_body<MODE, W8, 1, 4, W8 ? 4 : 8, W8 ? 3 : 2, F>(p, lds);
      else if constexpr (W8) gemm_stream_body<MODE, W8, 1, 2, 8, 2, F>(p, lds);
    };
    if (p.M <= (W8 ? 4 : 8)) forms(std::true_type{});
    else forms(std::false_type{});
  } else if constexpr (R == 2) {
    if (p.tile == 1) gemm_stream_body<MODE, W8, 2, 1, W8 ? 4 : 8, W8 ? 4 : 3>(p, lds);
    else if (p.tile == 2) gemm_stream_body<MODE, W8, 2, 2, W8 ? 4 : 8, W8 ? 3 : 2>(p, lds);
    else if constexpr (W8) gemm_stream_body<MODE, W8, 2, 3, 4, 2>(p, lds);
    else gemm_stream_body<MODE, W8, 2, 4, 4, 3>(p, lds);
  } else {
    if (p.tile == 1) gemm_stream_body<MODE, W8, 4, 1, W8 ? 4 : 8, 2>(p, lds);
    else if (W8 || p.tile == 2) gemm_stream_body<MODE, W8, 4, 2, 4, W8 ? 2 : 3>(p, lds);
    else if constexpr (!W8) gemm_stream_body<MODE, W8, 4, 4, 4, 2>(p, lds);
  }
}

// ------------------------------------------------------------ general GEMM
// 64x64 output tile, 256 threads, each 4x4 outputs; K in steps of 16 staged
// through LDS with bounds-checked element loads (zero fill past the edges).
template <bool INT8>
__device__ __forceinline__ void gemm_general_body(const GemmArgs& p) {
  __shared__ float As[16][64 + 1];
  __shared__ float Bs[16][64 + 1];
  __shared__ int Ai[16][64 + 1];
  __shared__ int Bi[16][64 + 1];
  const int tid = threadIdx.x;
  const int tm = blockIdx.x / p.tiles_n;
  const int tn = blockIdx.x % p.tiles_n;
  const int m0 = tm * 64, n0 = tn * 64;
  const int tx = tid & 15, ty = tid >> 4;  // 16 x 16 threads, 4x4 each
  float accf[4][4] = {};
  int acci[4][4] = {};
  for (int k0 = 0; k0 < p.K; k0 += 16) {
    for (int e = tid; e < 16 * 64; e += 256) {
      const int kk = e / 64, mm = e % 64;
      const int m = m0 + mm, k = k0 + kk;
      const bool inb = (m < p.M) && (k < p.K);
      const long long ia = (long long)m * p.a_s0 + (long long)k * p.a_s1;
      if (INT8) Ai[kk][mm] = !inb ? 0 : p.a_dtype == DT_UINT8 ? (int)((const uint8_t*)p.a)[ia]
                                                             : (int)((const int8_t*)p.a)[ia];
      else As[kk][mm] = inb ? load_as_f32(p.a, ia, p.a_dtype) : 0.0f;
      const int n = n0 + mm;
      const bool inbb = (n < p.N) && (k < p.K);
      const long long ib = (long long)k * p.b_s0 + (long long)n * p.b_s1;
      if (INT8) Bi[kk][mm] = !inbb ? 0 : p.b_dtype == DT_UINT8 ? (int)((const uint8_t*)p.b)[ib]
                                                               : (int)((const int8_t*)p.b)[ib];
      else if (p.b_dtype == DT_INT8) Bs[kk][mm] = inbb ? (float)((const int8_t*)p.b)[ib] : 0.0f;
      else Bs[kk][mm] = inbb ? load_as_f32(p.b, ib, p.b_dtype) : 0.0f;
    }
    __syncthreads();
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if (INT8) acci[i][j] = (int)((uint32_t)acci[i][j] + (uint32_t)(Ai[kk][ty * 4 + i] * Bi[kk][tx * 4 + j]));
          else accf[i][j] = fmaf(As[kk][ty * 4 + i], Bs[kk][tx * 4 + j], accf[i][j]);
        }
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int m = m0 + ty * 4 + i;
    if (m >= p.M) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = n0 + tx * 4 + j;
      if (n >= p.N) continue;
      float v;
      if (INT8) {
        if (p.acc_out) p.acc_out[(long long)m * p.acc_s0 + n] = acci[i][j];
        if (!p.sa) continue;
        v = ((float)acci[i][j] * p.sa[m]) * p.sb[n];
      } else {
        v = accf[i][j];
        if (p.bscale) v *= load_as_f32(p.bscale, n, p.bscale_dtype);
      }
      store_from_f32(p.c, (long long)m * p.c_s0 + (long long)n * p.c_s1, p.c_dtype, v);
    }
  }
}

}  // namespace g950

#define G950_GEMM_MFMA(NAME, MODE, WM, WN, UMASK, KT)                                        \
  extern "C" __global__ __launch_bounds__(WM * WN * 64) void NAME(const g950::GemmArgs p) {  \
    g950::gemm_mfma_body<MODE, WM, WN, UMASK, KT>(p);                                      \
  }
// row-major B [K, N] read directly (M, N >= 256, whole 64-k slabs; host checks)
#define G950_GEMM_MFMA_RB(NAME, MODE)                                                       \
  extern "C" __global__ __launch_bounds__(512) void NAME(const g950::GemmArgs p) {         \
    __shared__ __attribute__((aligned(1024))) char lds[4 * g950::BM * g950::SLAB];        \
    if (p.tile == g950::GEMM_TILE_128x128)                                                 \
      g950::gemm_tile_body<MODE, 128, 128, 0, 4, false, true>(p, lds);                     \
    else if (p.tile == g950::GEMM_TILE_64x128)                                             \
      g950::gemm_tile_body<MODE, 64, 128, 0, 5, false, true>(p, lds);                      \
    else if (p.tile == g950::GEMM_TILE_64x64)                                              \
      g950::gemm_tile_body<MODE, 64, 64, 0, 8, false, true>(p, lds);                       \
    else                                                                                   \
      g950::gemm_mfma16_body<MODE, 4, 2, 0, true>(p, lds);                                 \
  }
G950_GEMM_MFMA_RB(g950_gemm_bf16_256x256_rb, g950::GEMM_BF16)
G950_GEMM_MFMA_RB(g950_gemm_f16_256x256_rb, g950::GEMM_F16)
G950_GEMM_MFMA(g950_gemm_bf16_256x256, g950::GEMM_BF16, 4, 2, 0, false)
G950_GEMM_MFMA(g950_gemm_f16_256x256, g950::GEMM_F16, 4, 2, 0, false)
G950_GEMM_MFMA(g950_gemm_i8_256x256, g950::GEMM_I8, 4, 2, 0, false)
// K not a whole 128-byte slab (16-byte rows): the last slab's tail reads zeros
G950_GEMM_MFMA(g950_gemm_bf16_256x256_kt, g950::GEMM_BF16, 4, 2, 0, true)
G950_GEMM_MFMA(g950_gemm_f16_256x256_kt, g950::GEMM_F16, 4, 2, 0, true)
G950_GEMM_MFMA(g950_gemm_i8_256x256_kt, g950::GEMM_I8, 4, 2, 0, true)
// few rows of A: up to 16, 32 and 64
#define G950_FEW_ROWS(NAME, MODE, W8, R)                                                   \
  extern "C" __global__ __launch_bounds__(512) void NAME(const g950::GemmArgs p) {         \
    __shared__ __attribute__((aligned(1024))) char lds[g950::FEW_LDS];                     \
    g950::gemm_few_rows<MODE, W8, R>(p, lds);                                              \
  }
#define G950_GEMM_SKINNY(TY, MODE)                          \
  G950_FEW_ROWS(g950_gemm_skinny16_##TY, MODE, false, 1)    \
  G950_FEW_ROWS(g950_gemm_skinny32_##TY, MODE, false, 2)    \
  G950_FEW_ROWS(g950_gemm_skinny64_##TY, MODE, false, 4)
G950_GEMM_SKINNY(bf16, g950::GEMM_BF16)
G950_GEMM_SKINNY(f16, g950::GEMM_F16)
G950_GEMM_SKINNY(f32, g950::GEMM_F32)
G950_GEMM_SKINNY(i8, g950::GEMM_I8)
// int8 weights; _c16 and the plain name are one kernel: the names tell the
// two classes of grids that callers and tests know
#define G950_W8A16_SKINNY(TY, MODE)                                \
  G950_FEW_ROWS(g950_gemm_w8a16_skinny_##TY, MODE, true, 1)        \
  G950_FEW_ROWS(g950_gemm_w8a16_skinny_c16_##TY, MODE, true, 1)    \
  G950_FEW_ROWS(g950_gemm_w8a16_skinny32_##TY, MODE, true, 2)      \
  G950_FEW_ROWS(g950_gemm_w8a16_skinny64_##TY, MODE, true, 4)
G950_W8A16_SKINNY(bf16, g950::GEMM_BF16)
G950_W8A16_SKINNY(f16, g950::GEMM_F16)
// int8 weights, up to four rows of A, more columns than one round of the CUs
// holds: 32 columns per workgroup, two workgroups per CU.  One row of A (us;
// 64 columns and one workgroup per CU -> this; the register-loading kernel):
// 100000 x 4096 93.6 -> 65.3 (84.5), 50000 x 8192 93.8 -> 69.8 (74.5), 20000 x
// 4096 25.2 -> 17.6 (22.0).
#define G950_W8A16_FEW(TY, MODE)                                                                       \
  extern "C" __global__ __launch_bounds__(512) void g950_gemm_w8a16_few_##TY(const g950::GemmArgs p) { \
    __shared__ __attribute__((aligned(1024))) char lds[80 * 1024];                                     \
    g950::gemm_stream_body<MODE, true, 1, 2, 8, 2, true, false, true>(p, lds);                         \
  }
G950_W8A16_FEW(bf16, g950::GEMM_BF16)
G950_W8A16_FEW(f16, g950::GEMM_F16)
// int8 weights, rows out of 32-bit reach (the last token of long sequences):
// 32 columns per workgroup up to 64 rows of A, and the tiles.  The address
// arithmetic is hidden: 16 x 4096 x 8192 with A's rows 2^28 elements apart
// 11.0 us (10.5 at 2^26, in reach), 64 x 8192 x 8192 46, 512 x 4096 x 4096 36.
#define G950_W8A16_FAR(TY, MODE, ROWS, R, W, NS)                                                    \
  extern "C" __global__ __launch_bounds__(W * 64) void g950_gemm_w8a16_far##ROWS##_##TY(const g950::GemmArgs p) { \
    __shared__ __attribute__((aligned(1024))) char lds[g950::FEW_LDS];                              \
    g950::gemm_stream_body<MODE, true, R, 2, W, NS, false, true>(p, lds);                           \
  }
#define G950_W8A16_FARS(TY, MODE)              \
  G950_W8A16_FAR(TY, MODE, 16, 1, 8, 2)        \
  G950_W8A16_FAR(TY, MODE, 32, 2, 4, 3)        \
  G950_W8A16_FAR(TY, MODE, 64, 4, 4, 2)        \
  extern "C" __global__ __launch_bounds__(512) void g950_gemm_w8a16_far_##TY##_128x128(const g950::GemmArgs p) { \
    g950::gemm_w8a16_tiles<MODE, true>(p);     \
  }
G950_W8A16_FARS(bf16, g950::GEMM_BF16)
G950_W8A16_FARS(f16, g950::GEMM_F16)
extern "C" __global__ __launch_bounds__(256) void g950_transpose_b16(const g950::GemmArgs p) {
  g950::transpose16_body(p);
}
extern "C" __global__ __launch_bounds__(256) void g950_transpose_b32(const g950::GemmArgs p) {
  g950::transpose32_body(p);
}
extern "C" __global__ __launch_bounds__(256) void g950_transpose_b8(const g950::GemmArgs p) {
  g950::transpose8_body(p);
}
// fp32 on v_mfma_f32_32x32x2_f32 (the matmul corpus's base dtype)
G950_GEMM_MFMA(g950_gemm_f32_256x256, g950::GEMM_F32, 4, 2, 0, false)
G950_GEMM_MFMA(g950_gemm_f32_256x256_kt, g950::GEMM_F32, 4, 2, 0, true)
// int8 signedness variants of the reference family (a100c/plan/tiles.py:121-126):
// uint8 A x int8 B, int8 A x uint8 B, uint8 x uint8
G950_GEMM_MFMA(g950_gemm_u8s8_256x256, g950::GEMM_I8, 4, 2, 1, false)
G950_GEMM_MFMA(g950_gemm_s8u8_256x256, g950::GEMM_I8, 4, 2, 2, false)
G950_GEMM_MFMA(g950_gemm_u8u8_256x256, g950::GEMM_I8, 4, 2, 3, false)
extern "C" __global__ __launch_bounds__(256) void g950_i8_sums(const g950::I8SumArgs p) {
  g950::i8_sums_body(p);
}
// (128x128: the largest of its tiles)
extern "C" __global__ __launch_bounds__(512) void g950_gemm_w8a16_bf16_128x128(const g950::GemmArgs p) {
  g950::gemm_w8a16_tiles<g950::GEMM_BF16>(p);
}
extern "C" __global__ __launch_bounds__(512) void g950_gemm_w8a16_f16_128x128(const g950::GemmArgs p) {
  g950::gemm_w8a16_tiles<g950::GEMM_F16>(p);
}
extern "C" __global__ __launch_bounds__(256) void g950_gemm_general(const g950::GemmArgs p) {
  g950::gemm_general_body<false>(p);
}
extern "C" __global__ __launch_bounds__(256) void g950_gemm_general_i8(const g950::GemmArgs p) {
  g950::gemm_general_body<true>(p);
}
extern "C" __global__ __launch_bounds__(256) void g950_widen_i8_bf16(const g950::GemmArgs p) {
  g950::widen_i8_body<false>(p);
}
extern "C" __global__ __launch_bounds__(256) void g950_widen_i8_f16(const g950::GemmArgs p) {
  g950::widen_i8_body<true>(p);
}
