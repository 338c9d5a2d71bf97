// Whole-problem MFMA GEMM for gfx950 with a register-fused epilogue.
//
// Replaces the reference's "outer loops + brgemm microkernel call" structure
// (lib/gc/Transforms/DeepTileContractionOp.cpp:506-540 calling
// dnnl_brgemm_execute, lib/gc/ExecutionEngine/CPURuntime/Microkernel/
// BrgemmOnednn.cpp:145-168) by one kernel per matmul:
//   C[M,N] = epilogue( A[M,K] . B[K,N] ),  A and B plain row-major.
// ES = 2: bf16 x bf16 -> f32 accumulate (v_mfma_f32_32x32x16_bf16)
// ES = 1: (u8|s8) x s8 -> s32 accumulate (v_mfma_i32_32x32x32_i8)
//
// Workgroup tile 256 x 256, 128 bytes of K per stage (64 bf16 / 128 int8),
// 8 waves as 2 (M) x 4 (N), wave tile 128 x 64 = 4 x 2 MFMA tiles of 32 x 32.
// LDS: two stages of {A 256 rows x 128 B, B (128/ES) rows x 256*ES B} = 128 KiB.
//
// Operand roles are swapped on purpose: the MFMA's first operand is the B
// fragment (rows = n), the second the A fragment (columns = m).  The 32x32
// accumulator then gives every lane 4 consecutive n for one m, so the epilogue
// stores 8 (bf16) or 16 (f32/s32) contiguous bytes per lane and reads bias /
// scale / colsum as 4-vectors.
//
// B is row-major [K,N] (n contiguous) while the MFMA wants k-contiguous
// fragments: the transposition happens in the LDS read with
// ds_read_b64_tr_b16 / ds_read_b64_tr_b8, so the tile is stored exactly as it
// lies in memory.  This is the GPU analogue of the VNNI re-layout the
// reference's brgemm requires of B (lib/gc/Dialect/Microkernel/
// MicrokernelOps.cpp:380-389) without a separate packing pass.
//
// LDS swizzles (16-byte chunk index XOR):
//   A: chunk ^= (row >> 1) & 7        -> ds_read_b128 of 32 rows x 16 B is
//                                        conflict free over 64 banks
//   B: chunk ^= (krow % RG) * CW      -> RG = rows per transpose group (4 for
//                                        16-bit, 8 for 8-bit), CW = 16-byte
//                                        chunks one read touches per row
#pragma once
#include <type_traits>

#include "common.hpp"
#include "gemm_params.h"

namespace gcmi {

static constexpr int G_BM = 256, G_BN = 256, G_KBYTES = 128;
static constexpr int G_THREADS = 512;
static constexpr int G_STAGE_BYTES = 65536; // A 32 KiB + B 32 KiB
#ifndef G_FAST_WJ
// wave layout of the fast path: 2 = 8 waves of 128 x 64 (two per SIMD), 4 = 4 waves of 128 x 128 (one per
// SIMD, a third less LDS read traffic).  Measured on MI355X: the 4-wave layout is 5-7 % slower on bf16
// 4096^3 / 8192^3 and 19 % slower on the int8 MLP layer (nothing overlaps its epilogue), so 2 it is.
#define G_FAST_WJ 2
#endif
#ifndef G_FAST_KS
#define G_FAST_KS 2 // MFMA k-steps per LDS stage of the fast path: 2 (4-stage ring) or 4 (2-stage ring)
#endif

template <int ES> struct MfmaOp;
template <> struct MfmaOp<2> {
  typedef f32x16_t acc_t;
  typedef float acc_elem_t;
  static __device__ __forceinline__ acc_t run(const uint4 &a, const uint4 &b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c,
                                                   0, 0, 0);
  }
  // 8 bytes: k..k+3 of one n
  static __device__ __forceinline__ uint2 tr_read(const char *p) {
    bf16x4_t v = __builtin_amdgcn_ds_read_tr16_b64_v4bf16((GCMI_LDS bf16x4_t *)p);
    return __builtin_bit_cast(uint2, v);
  }
};
template <> struct MfmaOp<1> {
  typedef i32x16_t acc_t;
  typedef int acc_elem_t;
  static __device__ __forceinline__ acc_t run(const uint4 &a, const uint4 &b, acc_t c) {
    return __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4_t, a), __builtin_bit_cast(i32x4_t, b), c, 0,
                                                 0, 0);
  }
  // 8 bytes: k..k+7 of one n
  static __device__ __forceinline__ uint2 tr_read(const char *p) {
    i32x2_t v = __builtin_amdgcn_ds_read_tr8_b64_v2i32((GCMI_LDS i32x2_t *)p);
    return __builtin_bit_cast(uint2, v);
  }
};

// 16-byte chunk from global memory, zero filled outside [0,rows) x [0,row_bytes)
template <bool EDGE>
__device__ __forceinline__ uint4 load_chunk(const char *base, int64_t row, int64_t rows, int64_t col_byte,
                                            int64_t row_bytes, int64_t ld_bytes) {
  if (!EDGE) {
    return *reinterpret_cast<const uint4 *>(base + row * ld_bytes + col_byte);
  } else {
    uint4 v = make_uint4(0, 0, 0, 0);
    if (row >= rows || col_byte >= row_bytes)
      return v;
    const char *p = base + row * ld_bytes + col_byte;
    int64_t nvalid = row_bytes - col_byte;
    if (nvalid >= 16 && ((reinterpret_cast<uintptr_t>(p) & 15) == 0))
      return *reinterpret_cast<const uint4 *>(p);
    unsigned char tmp[16];
#pragma unroll
    for (int i = 0; i < 16; i++)
      tmp[i] = i < nvalid ? (unsigned char)p[i] : (unsigned char)0;
    v.x = tmp[0] | (tmp[1] << 8) | (tmp[2] << 16) | ((uint32_t)tmp[3] << 24);
    v.y = tmp[4] | (tmp[5] << 8) | (tmp[6] << 16) | ((uint32_t)tmp[7] << 24);
    v.z = tmp[8] | (tmp[9] << 8) | (tmp[10] << 16) | ((uint32_t)tmp[11] << 24);
    v.w = tmp[12] | (tmp[13] << 8) | (tmp[14] << 16) | ((uint32_t)tmp[15] << 24);
    return v;
  }
}

// Map a linear workgroup id to a tile so that the workgroups one XCD receives
// (hardware deals consecutive ids round-robin over 8 XCDs) cover a compact
// rectangle of tiles and share A/B panels in that XCD's L2.  Workgroups bid, bid + 8, ... take one run of tiles each; where
// their number is no multiple of 8 the first nblk % 8 runs are one longer (such numbers used to keep the hardware's order, every
// XCD then reads nearly every panel: a decoder layer's 1000 tokens, with 172 tiles of 256 x 256 each for gate and up, 415 us, now 392).
__device__ __forceinline__ int xcd_run(int bid, int nblk) {
  const int run = bid & 7;
  return run * (nblk >> 3) + min(run, nblk & 7) + (bid >> 3);
}
// tile `id` in groups of group_m tile rows, each walked column by column
__device__ __forceinline__ void tile_of_id(int id, int tiles_m, int tiles_n, int group_m, int &tm, int &tn) {
  int per_group = group_m * tiles_n;
  int g = id / per_group;
  int first_m = g * group_m;
  int gm = min(group_m, tiles_m - first_m);
  int in_g = id - g * per_group;
  tm = first_m + in_g % gm;
  tn = in_g / gm;
}
__device__ __forceinline__ void tile_of_block(int bid, int nblk, int tiles_m, int tiles_n, int group_m, int &tm,
                                              int &tn) {
  tile_of_id(xcd_run(bid, nblk), tiles_m, tiles_n, group_m, tm, tn);
}

// compile-time loop: the body receives std::integral_constant<int, I>, so every
// accumulator index is a constant and the accumulators stay in registers
template <int I, int N, typename F> __device__ __forceinline__ void static_for(F &&f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    static_for<I + 1, N>(f);
  }
}

template <int ACT> __device__ __forceinline__ float act_const(float x) { return apply_act(x, ACT); }

// two f32 -> two bf16 in one instruction (v_cvt_pk_bf16_f32: round to nearest even; not for NaNs, whose sign and
// payload it keeps); lo in bits 0-15
__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  typedef float f32x2_t __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
  const f32x2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}

// Epilogue shared by both kernels.  acc[j][i][r] holds
//   m = m0 + wm*128 + i*32 + (lane & 31),  n = n0 + wn*64 + j*32 + 8*(r/4) + 4*(lane >> 5) + r%4.
// Instantiated once per activation so that each copy unrolls completely.
// STAGED (whole tiles, bf16 output): the wave first lays its 128 x 64 result out
// in a private LDS region (rows of 128 B at a 144 B pitch), then reads it back
// row-wise so that every global store instruction writes eight complete
// 128-byte lines (16 B per lane) instead of 32 scattered 16-byte pieces.
static constexpr int G_STG_PITCH = 144;
static constexpr int G_STG_WAVE_BYTES = 128 * G_STG_PITCH; // 18 KiB per wave

// WJ = MFMA tiles along n per wave: 2 (8 waves as 2 x 4, wave tile 128 x 64) or 4
// (4 waves as 2 x 2, wave tile 128 x 128).
// LDSP (whole-tile kernels): the tile's 256 column parameters were laid out in LDS when the kernel started
// (colp[0..255] bias as f32, -0.0 when there is none; [256..511] scale; [512..767] comp * colsum as s32), so a
// lane fetches its four columns with one ds_read_b128 per array instead of scalar global loads behind a wait.
// MI16: the accumulators come from 16x16x32 MFMAs.  acc[j][i] still covers columns j*32.. and rows i*32.. of the wave
// tile, as four 16 x 16 tiles: elements 4q..4q+3 belong to the tile at columns 16*(q/2), rows 16*(q%2), where a
// lane holds columns 4*(lane/16)..+3 of row lane%16.
template <int ES, bool EDGE, int ACT, bool STAGED, int WJ = 2, bool LDSP = false, bool MI16 = false>
__device__ __forceinline__ void gemm_epilogue_act(const GemmParams &p, typename MfmaOp<ES>::acc_t (&acc)[WJ][4],
                                                  int64_t m0, int64_t n0, int wm, int wn, int l32, int lh,
                                                  char *stg, const float *colp = nullptr) {
  constexpr int PITCH = 64 * WJ + 16; // staging row: 32*WJ bf16 + 16 bytes of padding
  const int out_dt = STAGED ? (int)DT_BF16 : p.out_dt; // only bf16 results are staged
  const int out_es = out_dt == DT_BF16 ? 2 : 4;
  char *Cb = reinterpret_cast<char *>(p.C);
  static_for<0, WJ>([&](auto jc) {
    constexpr int j = decltype(jc)::value;
    static_for<0, 4>([&](auto qc) {
      constexpr int q = decltype(qc)::value;
      // this lane's four columns and its row inside the 32 x 32 block (j, i)
      const int n_off = MI16 ? 16 * (q >> 1) + 4 * (2 * lh + (l32 >> 4)) : 8 * q + 4 * lh;
      const int m_off = MI16 ? 16 * (q & 1) + (l32 & 15) : l32;
      const int64_t n = n0 + wn * (32 * WJ) + j * 32 + n_off;
      float bias4[4] = {0.f, 0.f, 0.f, 0.f}, scale4[4] = {1.f, 1.f, 1.f, 1.f};
      int cs4[4] = {0, 0, 0, 0}; // comp * colsum
      if constexpr (LDSP) {
        const int col = wn * (32 * WJ) + j * 32 + n_off;
        const f32x4_t b = *reinterpret_cast<const f32x4_t *>(colp + col);
        bias4[0] = b[0], bias4[1] = b[1], bias4[2] = b[2], bias4[3] = b[3];
        if (ES == 1) {
          const f32x4_t sc = *reinterpret_cast<const f32x4_t *>(colp + 256 + col);
          const i32x4_t cs = *reinterpret_cast<const i32x4_t *>(colp + 512 + col);
          scale4[0] = sc[0], scale4[1] = sc[1], scale4[2] = sc[2], scale4[3] = sc[3];
          cs4[0] = cs[0], cs4[1] = cs[1], cs4[2] = cs[2], cs4[3] = cs[3];
        }
      } else {
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (!EDGE || n + e < p.N) {
            if (p.bias)
              bias4[e] = p.bias_dt == DT_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p.bias)[n + e])
                                              : reinterpret_cast<const float *>(p.bias)[n + e];
            if (ES == 1) {
              if (p.scale)
                scale4[e] = p.scale[n + e];
              if (p.colsum)
                cs4[e] = p.comp * p.colsum[n + e];
            }
          }
        }
      }
      static_for<0, 4>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int64_t m = m0 + wm * 128 + i * 32 + m_off;
        if (EDGE && m >= p.M)
          return;
        uint32_t o32[4];
        uint16_t o16[4];
        float xf[4] = {0.f, 0.f, 0.f, 0.f};
        float res4[4] = {0.f, 0.f, 0.f, 0.f};
        if (ES == 2 && p.residual) {
          const int64_t at = m * p.ldr + n;
          if (!EDGE) { // the launcher sends unaligned residuals to the EDGE kernels
            if (p.residual_dt == DT_BF16) {
              const uint2 v = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint16_t *>(p.residual) + at);
              res4[0] = __uint_as_float(v.x << 16), res4[1] = __uint_as_float(v.x & 0xffff0000u);
              res4[2] = __uint_as_float(v.y << 16), res4[3] = __uint_as_float(v.y & 0xffff0000u);
            } else {
              const f32x4_t v = *reinterpret_cast<const f32x4_t *>(reinterpret_cast<const float *>(p.residual) + at);
              res4[0] = v[0], res4[1] = v[1], res4[2] = v[2], res4[3] = v[3];
            }
          } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
              if (n + e < p.N)
                res4[e] = p.residual_dt == DT_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p.residual)[at + e])
                                                   : reinterpret_cast<const float *>(p.residual)[at + e];
          }
        }
        if constexpr (ES == 2 && LDSP && STAGED) {
          // bf16 graph, whole tiles: the same rounding points as below (after the matmul and after every bf16 op,
          // lib/gc/Transforms/Pipeline.cpp:79-95), rounded in pairs by v_cvt_pk_bf16_f32.  A NaN stays a NaN
          // through the ops that follow, so only the last conversion has to give it the reference's 0x7FC0.
          float x[4] = {(float)acc[j][i][4 * q], (float)acc[j][i][4 * q + 1], (float)acc[j][i][4 * q + 2],
                        (float)acc[j][i][4 * q + 3]};
          uint32_t p0, p1;
          auto rnd = [&]() {
            p0 = pack_bf16x2(x[0], x[1]), p1 = pack_bf16x2(x[2], x[3]);
            x[0] = __uint_as_float(p0 << 16), x[1] = __uint_as_float(p0 & 0xffff0000u);
            x[2] = __uint_as_float(p1 << 16), x[3] = __uint_as_float(p1 & 0xffff0000u);
          };
          rnd();
          if (p.bias) {
#pragma unroll
            for (int e = 0; e < 4; e++)
              x[e] = x[e] + bias4[e];
            rnd();
          }
          if (ACT != ACT_NONE) {
#pragma unroll
            for (int e = 0; e < 4; e++)
              x[e] = apply_act_of_bf16(x[e], ACT);
            if (ACT == ACT_RELU) { // max(x, 0) of a bf16 value is a bf16 value: nothing to round
              p0 = (__float_as_uint(x[0]) >> 16) | (__float_as_uint(x[1]) & 0xffff0000u);
              p1 = (__float_as_uint(x[2]) >> 16) | (__float_as_uint(x[3]) & 0xffff0000u);
            } else {
              rnd();
            }
          }
          if (p.residual) {
#pragma unroll
            for (int e = 0; e < 4; e++)
              x[e] = x[e] + res4[e];
            rnd();
          }
          const float any_nan = (x[0] + x[1]) + (x[2] + x[3]); // a NaN if one of them is (or opposite infinities)
          if (__builtin_expect(any_nan != any_nan, 0)) {
            if (x[0] != x[0]) p0 = (p0 & 0xffff0000u) | 0x7FC0u;
            if (x[1] != x[1]) p0 = (p0 & 0x0000ffffu) | 0x7FC00000u;
            if (x[2] != x[2]) p1 = (p1 & 0xffff0000u) | 0x7FC0u;
            if (x[3] != x[3]) p1 = (p1 & 0x0000ffffu) | 0x7FC00000u;
          }
          *reinterpret_cast<uint2 *>(stg + (i * 32 + m_off) * PITCH + (j * 32 + n_off) * 2) = make_uint2(p0, p1);
          return;
        }
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if (ES == 1) {
            // s32 accumulator of (a ^ 0x80) * w; comp restores / applies the
            // zero-point term in exact integer arithmetic.
            int c = (int)acc[j][i][4 * q + e] + cs4[e];
            if (out_dt == DT_S32) {
              o32[e] = (uint32_t)c;
              o16[e] = 0;
            } else {
              float x;
              if constexpr (LDSP) { // an absent bias is -0.0: the fused multiply-add then equals the product
                x = fmaf((float)c, scale4[e], bias4[e]);
              } else {
                x = (float)c * scale4[e];
                if (p.bias)
                  x = x + bias4[e];
              }
              x = act_const<ACT>(x);
              o32[e] = __float_as_uint(x);
              if constexpr (LDSP && STAGED)
                xf[e] = x; // converted in pairs below
              else
                o16[e] = f32_to_bf16_bits(x);
            }
          } else {
            float x = (float)acc[j][i][4 * q + e];
            const float r = res4[e];
            if (out_dt == DT_BF16) {
              // bf16 graph: round after the matmul and after every bf16 op
              // (lib/gc/Transforms/Pipeline.cpp:79-95)
              x = round_bf16(x);
              if (p.bias)
                x = round_bf16(x + bias4[e]);
              if (ACT != ACT_NONE)
                x = round_bf16(apply_act_of_bf16(x, ACT));
              if (p.residual)
                x = round_bf16(x + r);
              o16[e] = f32_to_bf16_bits(x);
              o32[e] = 0;
            } else {
              if (p.bias)
                x = x + bias4[e];
              x = act_const<ACT>(x);
              if (p.residual) { // kept apart from the activation's last multiply: the sum equals a separate add
#pragma clang fp contract(off)
                x = x + r;
              }
              o32[e] = __float_as_uint(x);
              o16[e] = 0;
            }
          }
        }
        if (STAGED) {
          uint2 packed;
          if constexpr (LDSP && ES == 1) {
            // v_cvt_pk_bf16_f32 rounds to nearest even like the scalar routine but keeps a NaN's sign (the
            // hardware's own invalid-operation NaN is negative), so four values with a NaN among them (their sum
            // is one; so is the sum of opposite infinities) take the scalar routine: NaN -> 0x7FC0
            const float any_nan = (xf[0] + xf[1]) + (xf[2] + xf[3]);
            if (__builtin_expect(any_nan != any_nan, 0))
              packed = make_uint2(f32_to_bf16_bits(xf[0]) | ((uint32_t)f32_to_bf16_bits(xf[1]) << 16),
                                  f32_to_bf16_bits(xf[2]) | ((uint32_t)f32_to_bf16_bits(xf[3]) << 16));
            else
              packed = make_uint2(pack_bf16x2(xf[0], xf[1]), pack_bf16x2(xf[2], xf[3]));
          } else {
            packed = make_uint2(o16[0] | ((uint32_t)o16[1] << 16), o16[2] | ((uint32_t)o16[3] << 16));
          }
          *reinterpret_cast<uint2 *>(stg + (i * 32 + m_off) * PITCH + (j * 32 + n_off) * 2) = packed;
          return;
        }
        char *dst = Cb + (m * p.ldc + n) * out_es;
        if (!EDGE) {
          if (out_es == 2)
            *reinterpret_cast<uint2 *>(dst) =
                make_uint2(o16[0] | ((uint32_t)o16[1] << 16), o16[2] | ((uint32_t)o16[3] << 16));
          else
            *reinterpret_cast<uint4 *>(dst) = make_uint4(o32[0], o32[1], o32[2], o32[3]);
        } else {
#pragma unroll
          for (int e = 0; e < 4; e++) {
            if (n + e < p.N) {
              if (out_es == 2)
                reinterpret_cast<uint16_t *>(dst)[e] = o16[e];
              else
                reinterpret_cast<uint32_t *>(dst)[e] = o32[e];
            }
          }
        }
      });
    });
  });
  if (STAGED) {
    // wave-private region: only this wave's own LDS writes have to land
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    const int lane = lh * 32 + l32;
    constexpr int LPR = 4 * WJ, RPP = 64 / LPR; // lanes per row (16 B each), rows per pass
    const int rr = lane / LPR, cc = lane % LPR;
#pragma unroll
    for (int it = 0; it < 128 / RPP; it++) {
      const int row = it * RPP + rr;
      uint4 v = *reinterpret_cast<const uint4 *>(stg + row * PITCH + cc * 16);
      typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
      u32x4_t vv = {v.x, v.y, v.z, v.w};
      __builtin_nontemporal_store(vv, reinterpret_cast<u32x4_t *>(Cb + ((m0 + wm * 128 + row) * p.ldc + n0 + wn * (32 * WJ) + cc * 8) * 2));
    }
  }
}

template <int ES, bool EDGE, bool STAGED, int WJ = 2, bool LDSP = false, bool MI16 = false>
__device__ __forceinline__ void gemm_epilogue(const GemmParams &p, typename MfmaOp<ES>::acc_t (&acc)[WJ][4], int64_t m0,
                                              int64_t n0, int wm, int wn, int l32, int lh, char *stg,
                                              const float *colp = nullptr) {
  switch (p.act) {
  case ACT_RELU:
    gemm_epilogue_act<ES, EDGE, ACT_RELU, STAGED, WJ, LDSP, MI16>(p, acc, m0, n0, wm, wn, l32, lh, stg, colp);
    break;
  case ACT_GELU_ERF:
    gemm_epilogue_act<ES, EDGE, ACT_GELU_ERF, STAGED, WJ, LDSP, MI16>(p, acc, m0, n0, wm, wn, l32, lh, stg, colp);
    break;
  case ACT_GELU_TANH:
    gemm_epilogue_act<ES, EDGE, ACT_GELU_TANH, STAGED, WJ, LDSP, MI16>(p, acc, m0, n0, wm, wn, l32, lh, stg, colp);
    break;
  case ACT_SIGMOID:
    gemm_epilogue_act<ES, EDGE, ACT_SIGMOID, STAGED, WJ, LDSP, MI16>(p, acc, m0, n0, wm, wn, l32, lh, stg, colp);
    break;
  default:
    gemm_epilogue_act<ES, EDGE, ACT_NONE, STAGED, WJ, LDSP, MI16>(p, acc, m0, n0, wm, wn, l32, lh, stg, colp);
    break;
  }
}

// TB: B is stored [N,K] (k contiguous).  Its tile then has the geometry of the A tile (256 rows x 128 bytes of K),
// takes the same swizzle, and its fragments are plain 16-byte reads like A's: no transposing LDS read is needed.
template <int ES, bool EDGE, bool TB = false> __global__ __launch_bounds__(G_THREADS) void gemm_tile256_kernel(GemmParams p) {
  typedef MfmaOp<ES> Op;
  typedef typename Op::acc_t acc_t;
  constexpr int BK = G_KBYTES / ES;        // K elements per stage
  constexpr int B_ROW_BYTES = G_BN * ES;   // bytes per k-row of the B tile
  constexpr int B_CPR = B_ROW_BYTES / 16;  // 16-byte chunks per B row
  constexpr int RG = ES == 2 ? 4 : 8;      // k-rows per transpose-read group
  constexpr int CW = ES == 2 ? 4 : 2;      // chunks per row one transpose read spans
  constexpr int KSTEP = 32 / ES;           // K elements one MFMA consumes

  __shared__ __align__(16) char smem[2 * G_STAGE_BYTES];

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 2, wn = wave & 3;
  const int l32 = lane & 31, lh = lane >> 5;

  const int tiles_m = (int)((p.M + G_BM - 1) / G_BM), tiles_n = (int)((p.N + G_BN - 1) / G_BN);
  int tm, tn;
  tile_of_block(blockIdx.x, gridDim.x, tiles_m, tiles_n, p.group_m, tm, tn);
  const int64_t m0 = (int64_t)tm * G_BM, n0 = (int64_t)tn * G_BN;

  const int64_t lda_b = p.lda * ES, ldb_b = p.ldb * ES;
  const int64_t bz = blockIdx.y; // batch
  const char *Ab = reinterpret_cast<const char *>(p.A) + bz * p.a_bs * ES;
  const char *Bb = reinterpret_cast<const char *>(p.B) + bz * p.b_bs * ES;
  p.C = reinterpret_cast<char *>(p.C) + bz * p.c_bs * (p.out_dt == DT_BF16 ? 2 : 4);
  if (p.residual)
    p.residual = reinterpret_cast<const char *>(p.residual) + bz * p.c_bs * (p.residual_dt == DT_BF16 ? 2 : 4);

  // ---- global -> register staging assignment: 4 A chunks + 4 B chunks per thread
  const int a_row0 = tid >> 3, a_c = tid & 7;             // rows a_row0 + 64*i
  const int b_row0 = tid / B_CPR, b_c = tid % B_CPR;      // rows b_row0 + (512/B_CPR)*i
  constexpr int B_ROW_STEP = G_THREADS / B_CPR;
  uint32_t a_st[4], b_st[4]; // LDS store offsets inside a stage
#pragma unroll
  for (int i = 0; i < 4; i++) {
    int row = a_row0 + 64 * i;
    a_st[i] = row * 128 + ((a_c ^ ((row >> 1) & 7)) << 4);
    int krow = b_row0 + B_ROW_STEP * i;
    b_st[i] = TB ? 32768 + a_st[i] : 32768 + krow * B_ROW_BYTES + ((b_c ^ ((krow % RG) * CW)) << 4);
  }

  // ---- LDS read offsets of this lane's MFMA fragments
  const int sw = (l32 >> 1) & 7;
  uint32_t a_ld[4]; // per k-step chunk offset; + lane row base + i*4096
#pragma unroll
  for (int ks = 0; ks < 4; ks++)
    a_ld[ks] = (wm * 128 + l32) * 128 + (((2 * ks + lh) ^ sw) << 4);
  const int g = lane >> 4, i16 = lane & 15;
  uint32_t b_ld[2]; // + ks*8192 + jj*2048
  {
    const int kk = ES == 2 ? (i16 >> 2) : (i16 >> 1);
    const int cc = ES == 2 ? (i16 & 3) : (i16 & 1);
#pragma unroll
    for (int j = 0; j < 2; j++) {
      int chunk = ES == 2 ? (wn * 8 + j * 4 + 2 * (g & 1) + (cc >> 1)) : (wn * 4 + j * 2 + (g & 1));
      int sub = ES == 2 ? (cc & 1) * 8 : cc * 8;
      int krow_lane = (ES == 2 ? 8 : 16) * (g >> 1) + kk;
      b_ld[j] = 32768 + krow_lane * B_ROW_BYTES + ((chunk ^ (kk * CW)) << 4) + sub;
      if (TB) // row of the tile; + the k-step's chunk (swizzled like A's)
        b_ld[j] = 32768 + (wn * 64 + j * 32 + l32) * 128;
    }
  }

  acc_t acc[2][4];
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int r = 0; r < 16; r++)
        acc[j][i][r] = 0;

  const int64_t k_bytes = p.K * ES;
  const int KT = (int)((p.K + BK - 1) / BK);
  uint4 ra[4], rb[4];

  auto gload = [&](int kt) {
    const int64_t kb = (int64_t)kt * G_KBYTES; // byte offset along K of A
#pragma unroll
    for (int i = 0; i < 4; i++)
      ra[i] = load_chunk<EDGE>(Ab, m0 + a_row0 + 64 * i, p.M, kb + a_c * 16, k_bytes, lda_b);
#pragma unroll
    for (int i = 0; i < 4; i++)
      rb[i] = TB ? load_chunk<EDGE>(Bb, n0 + a_row0 + 64 * i, p.N, kb + a_c * 16, k_bytes, ldb_b)
                 : load_chunk<EDGE>(Bb, (int64_t)kt * BK + b_row0 + B_ROW_STEP * i, p.K, n0 * ES + b_c * 16,
                                    p.N * ES, ldb_b);
  };
  auto lstore = [&](int stage) {
    char *s = smem + stage * G_STAGE_BYTES;
    const uint32_t x = p.a_xor;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      uint4 v = ra[i];
      if (ES == 1) { // u8 activations: a - 128 as s8 == a ^ 0x80
        v.x ^= x;
        v.y ^= x;
        v.z ^= x;
        v.w ^= x;
      }
      *reinterpret_cast<uint4 *>(s + a_st[i]) = v;
    }
#pragma unroll
    for (int i = 0; i < 4; i++)
      *reinterpret_cast<uint4 *>(s + b_st[i]) = rb[i];
  };

  gload(0);
  lstore(0);
  __syncthreads();

  for (int kt = 0; kt < KT; kt++) {
    const int cur = kt & 1;
    if (kt + 1 < KT)
      gload(kt + 1);
    const char *s = smem + cur * G_STAGE_BYTES;
#pragma unroll
    for (int ks = 0; ks < 4; ks++) {
      uint4 af[4], bf[2];
#pragma unroll
      for (int i = 0; i < 4; i++)
        af[i] = *reinterpret_cast<const uint4 *>(s + a_ld[ks] + i * 4096);
#pragma unroll
      for (int j = 0; j < 2; j++) {
        if (TB) {
          bf[j] = *reinterpret_cast<const uint4 *>(s + b_ld[j] + (((2 * ks + lh) ^ sw) << 4));
        } else {
          uint2 lo = Op::tr_read(s + b_ld[j] + ks * 8192);
          uint2 hi = Op::tr_read(s + b_ld[j] + ks * 8192 + 2048);
          bf[j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
        }
      }
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 4; i++)
          acc[j][i] = Op::run(bf[j], af[i], acc[j][i]);
    }
    if (kt + 1 < KT)
      lstore(cur ^ 1);
    __syncthreads();
  }
  (void)KSTEP;

  gemm_epilogue<ES, EDGE, false>(p, acc, m0, n0, wm, wn, l32, lh, nullptr);
}

// ---------------------------------------------------------------------------
// Fast path: every dimension a multiple of the tile, 16-byte aligned operands.
//  * K is consumed in stages of KS MFMA k-steps (KS*32 bytes of K per row); the
//    LDS holds a ring of NST = 8/KS such stages (KS=2: 4 x 32 KiB, KS=4:
//    2 x 64 KiB).  Stage kt+NST-1 is requested while stage kt is computed, so
//    two to three stages of global->LDS traffic are always in flight: a CU's
//    L2->LDS path only delivers ~100 GB/s and has to stream without gaps.
//  * global -> LDS goes through global_load_lds_dwordx4: each wave instruction
//    drops 1 KiB straight into LDS (lane l at base + 16*l), no staging
//    registers and no ds_write.  The swizzle is applied on the GLOBAL side: the
//    lane that fills physical chunk P fetches logical chunk P ^ f(row).
//  * MFMA fragments are double buffered in registers: the LDS reads of k-step
//    s+1 are issued in the shadow of the MFMAs of k-step s, interleaved 1:1 by
//    the scheduler hints; the reads of the next stage's first k-step are issued
//    right after the stage barrier, under the last 8 MFMAs of the stage.
//  * The stage loop is unrolled over the ring, so every LDS address is static.
#define GCMI_GLB __attribute__((address_space(1)))

// SPLIT (split-K on a short A): only the first `mi` 32-row tiles of a wave hold rows of A; the others are
// neither read from LDS nor multiplied.
// TB (B stored [N,K]): the B tile is staged and read exactly like the A tile.
template <int ES, int KS, int WJ = 2, bool SPLIT = false, bool TB = false> struct FastGemm {
  static constexpr int NWAVES = 16 / WJ; // 8 or 4
  int mi = 4;
  typedef MfmaOp<ES> Op;
  typedef typename Op::acc_t acc_t;
  static constexpr int NST = 8 / KS;                  // stages in the LDS ring
  static constexpr int KB = KS * 32;                  // bytes of K per A row per stage
  static constexpr int BK = KB / ES;                  // K elements per stage
  static constexpr int A_BYTES = G_BM * KB;           // 16 or 32 KiB
  static constexpr int STAGE_BYTES = 2 * A_BYTES;     // B tile has the same size
  static constexpr int A_CPR = KB / 16;               // 16-byte chunks per A row: 4 or 8
  static constexpr int A_ROWS_PER_DMA = 1024 / KB;    // 16 or 8
  static constexpr int B_ROW_BYTES = G_BN * ES;
  static constexpr int RG = ES == 2 ? 4 : 8;
  static constexpr int CW = ES == 2 ? 4 : 2;
  static constexpr int B_ROWS_PER_DMA = 1024 / B_ROW_BYTES; // 2 (bf16) or 4 (int8)
  static constexpr int B_CPR = B_ROW_BYTES / 16;
  static constexpr int NDMA = KS * 8 / NWAVES;        // DMA instructions per operand per wave per stage

  static __device__ __forceinline__ int a_swz(int row) { return KS == 4 ? ((row >> 1) & 7) : ((row >> 2) & 3); }

  uint32_t a_src[NDMA], b_src[NDMA]; // per-lane byte offsets of this wave's DMA instructions
  uint32_t a_ld[KS], b_ld[TB ? KS : WJ]; // fragment read offsets
  uint32_t a_xor;
  int wave_u; // wave id, wave-uniform

  __device__ __forceinline__ void issue_loads(char *__restrict__ stage, const char *a_base, const char *b_base) const {
#pragma unroll
    for (int i = 0; i < NDMA; i++)
      __builtin_amdgcn_global_load_lds((GCMI_GLB const void *)(a_base + a_src[i]),
                                       (GCMI_LDS void *)(stage + (wave_u * NDMA + i) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < NDMA; i++)
      __builtin_amdgcn_global_load_lds((GCMI_GLB const void *)(b_base + b_src[i]),
                                       (GCMI_LDS void *)(stage + A_BYTES + (wave_u * NDMA + i) * 1024), 16, 0, 0);
  }

  __device__ __forceinline__ void load_frags(const char *__restrict__ s, int ks, uint4 (&af)[4], uint4 (&bf)[WJ]) const {
    if (SPLIT && mi == 0)
      return;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (SPLIT && i >= mi)
        break;
      uint4 v = *reinterpret_cast<const uint4 *>(s + a_ld[ks] + i * 32 * KB);
      if (ES == 1) // u8 activations: a - 128 as s8 == a ^ 0x80
        v = make_uint4(v.x ^ a_xor, v.y ^ a_xor, v.z ^ a_xor, v.w ^ a_xor);
      af[i] = v;
    }
#pragma unroll
    for (int j = 0; j < WJ; j++) {
      if (TB) {
        bf[j] = *reinterpret_cast<const uint4 *>(s + A_BYTES + b_ld[ks] + j * 32 * KB);
      } else {
        uint2 lo = Op::tr_read(s + b_ld[j] + ks * 8192);
        uint2 hi = Op::tr_read(s + b_ld[j] + ks * 8192 + 2048);
        bf[j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
    }
  }

  __device__ __forceinline__ void mfma_all(acc_t (&acc)[WJ][4], const uint4 (&af)[4], const uint4 (&bf)[WJ]) const {
#pragma unroll
    for (int j = 0; j < WJ; j++)
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (!SPLIT || i < mi)
          acc[j][i] = Op::run(bf[j], af[i], acc[j][i]);
  }

  // ask the scheduler for MFMA, DS read, MFMA, DS read, ... over the region
  static __device__ __forceinline__ void interleave_hint() {
    if (SPLIT)
      return;
    // the fragment reads of the next k-step go out with the first MFMAs, two per MFMA, so that they have landed
    // when the group ends and the wait in front of the next group finds little outstanding (1-4 % over one read
    // per MFMA spread over the whole group)
    constexpr int N_DS = 4 + (TB ? WJ : 2 * WJ);
    static_for<0, 4 * WJ>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0); // 1 MFMA
      constexpr int left = N_DS - 2 * i;
      if constexpr (left > 0)
        __builtin_amdgcn_sched_group_barrier(0x100, left < 2 ? left : 2, 0); // DS reads
    });
  }

  // wait until at most BEHIND later stages of this wave's DMA are still in flight
  // (and all of its LDS reads have returned)
  template <int BEHIND> static __device__ __forceinline__ void wait_dma() {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(BEHIND * 2 * NDMA) : "memory");
  }

  // One stage, branch free.  `cur` holds k-block kt (landed and barriered;
  // fragments of its k-step 0 are in a0/b0); the DMA of k-block kt+NST-1 goes
  // into `fill`, the buffer that was computed from one stage ago; `nxt` holds
  // k-block kt+1, behind which BEHIND more blocks are in flight.
  template <bool HAS_FILL, bool HAS_NEXT, int BEHIND>
  __device__ __forceinline__ void stage(char *__restrict__ cur, char *__restrict__ nxt, char *__restrict__ fill,
                                        const char *a_fill, const char *b_fill, acc_t (&acc)[WJ][4], uint4 (&a0)[4],
                                        uint4 (&b0)[WJ], uint4 (&a1)[4], uint4 (&b1)[WJ]) const {
    if (HAS_FILL)
      issue_loads(fill, a_fill, b_fill);
#pragma unroll
    for (int ks = 0; ks + 1 < KS; ks++) {
      if (ks & 1) {
        load_frags(cur, ks + 1, a0, b0);
        mfma_all(acc, a1, b1);
      } else {
        load_frags(cur, ks + 1, a1, b1);
        mfma_all(acc, a0, b0);
      }
      interleave_hint();
    }
    // every wave has its last fragments of `cur` in registers and its share of
    // k-block kt+1 landed in `nxt` before anyone moves on
    wait_dma<BEHIND>();
    __builtin_amdgcn_s_barrier();
    // with a 2-stage ring the next block lives in the buffer just filled: read it
    // through the same pointer the DMA was issued with
    if (HAS_NEXT)
      load_frags(NST == 2 ? fill : nxt, 0, a0, b0);
    mfma_all(acc, a1, b1);
    interleave_hint();
  }
};

template <int ES, int KS, int WJ, bool SPLIT = false, bool TB = false>
__global__ __launch_bounds__(1024 / WJ, 1) void gemm_tile256_fast_kernel(GemmParams p) {
  typedef FastGemm<ES, KS, WJ, SPLIT, TB> FG;
  typedef typename FG::acc_t acc_t;
  constexpr int NST = FG::NST;
  // ring of NST stages (128 KiB); the epilogue reuses the whole array as 8 x 18 KiB staging regions
  // behind them the tile's column parameters for the epilogue: bias, scale, comp * colsum (see gemm_epilogue_act).
  // One array on purpose: with a second LDS variable in the kernel the compiler puts a full vmcnt(0) wait in
  // front of the fragment reads of every stage (it then treats every LDS read as a reader of the DMA's target).
  __shared__ __align__(1024) char smem[8 * G_STG_WAVE_BYTES + (SPLIT ? 0 : 3 * G_BN * 4)];
  float *colp = reinterpret_cast<float *>(smem + 8 * G_STG_WAVE_BYTES);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = WJ == 2 ? wave >> 2 : wave >> 1, wn = WJ == 2 ? wave & 3 : wave & 1;
  const int l32 = lane & 31, lh = lane >> 5;

  const int tiles_m = (int)((p.M + G_BM - 1) / G_BM), tiles_n = (int)(p.N / G_BN);
  int tm, tn, slice = 0;
  if (SPLIT) { // the tiles of one K slice are neighbours in the grid; K slice = blockIdx / tiles
    const int tiles = tiles_m * tiles_n, tile = (int)blockIdx.x % tiles;
    tm = tile / tiles_n;
    tn = tile % tiles_n;
    slice = (int)blockIdx.x / tiles;
  } else {
    tile_of_block(blockIdx.x, gridDim.x, tiles_m, tiles_n, p.group_m, tm, tn);
  }
  const int64_t m0 = (int64_t)tm * G_BM, n0 = (int64_t)tn * G_BN;
  const int64_t lda_b = p.lda * ES, ldb_b = p.ldb * ES;
  if (!SPLIT) { // strided batch in blockIdx.y
    const int64_t bz = blockIdx.y;
    p.A = reinterpret_cast<const char *>(p.A) + bz * p.a_bs * ES;
    p.B = reinterpret_cast<const char *>(p.B) + bz * p.b_bs * ES;
    p.C = reinterpret_cast<char *>(p.C) + bz * p.c_bs * (p.out_dt == DT_BF16 ? 2 : 4);
  if (p.residual)
    p.residual = reinterpret_cast<const char *>(p.residual) + bz * p.c_bs * (p.residual_dt == DT_BF16 ? 2 : 4);
  }

  FG g;
  g.wave_u = wave;
  if (SPLIT) { // 32-row tiles of this wave that hold rows of A
    const int64_t left = p.M - m0 - wm * 128;
    g.mi = left <= 0 ? 0 : (int)min((int64_t)4, (left + 31) / 32);
  }
  g.a_xor = p.a_xor;
#pragma unroll
  for (int i = 0; i < FG::NDMA; i++) {
    // A: this instruction fills 1 KiB = A_ROWS_PER_DMA rows; lane -> (row, physical chunk)
    int row = (wave * FG::NDMA + i) * FG::A_ROWS_PER_DMA + lane / FG::A_CPR;
    int c = (lane % FG::A_CPR) ^ FG::a_swz(row);
    // rows past M (split-K on a short A): fetch the last row instead, its results are dropped
    const int row_src = (int)min((int64_t)row, p.M - 1 - m0);
    g.a_src[i] = (uint32_t)(row_src * lda_b + c * 16);
    // B: B_ROWS_PER_DMA k-rows; lane -> (krow, physical chunk)
    int krow = (wave * FG::NDMA + i) * FG::B_ROWS_PER_DMA + lane / FG::B_CPR;
    int cb = (lane % FG::B_CPR) ^ ((krow % FG::RG) * FG::CW);
    g.b_src[i] = TB ? (uint32_t)(row * ldb_b + c * 16) : (uint32_t)(krow * ldb_b + cb * 16);
  }
#pragma unroll
  for (int ks = 0; ks < KS; ks++) {
    int row = wm * 128 + l32; // + i*32: a multiple of 32 leaves the swizzle unchanged
    g.a_ld[ks] = row * FG::KB + (((2 * ks + lh) ^ FG::a_swz(row)) << 4);
  }
  {
    const int gq = lane >> 4, i16 = lane & 15;
    const int kk = ES == 2 ? (i16 >> 2) : (i16 >> 1);
    const int cc = ES == 2 ? (i16 & 3) : (i16 & 1);
    if constexpr (TB) {
#pragma unroll
      for (int ks = 0; ks < KS; ks++) {
        int row = wn * 32 * WJ + l32; // + j*32
        g.b_ld[ks] = row * FG::KB + (((2 * ks + lh) ^ FG::a_swz(row)) << 4);
      }
    } else {
#pragma unroll
      for (int j = 0; j < WJ; j++) {
        const int nb = wn * WJ + j; // 32-column block of the tile
        int chunk = ES == 2 ? (nb * 4 + 2 * (gq & 1) + (cc >> 1)) : (nb * 2 + (gq & 1));
        int sub = ES == 2 ? (cc & 1) * 8 : cc * 8;
        int krow_lane = (ES == 2 ? 8 : 16) * (gq >> 1) + kk;
        g.b_ld[j] = FG::A_BYTES + krow_lane * FG::B_ROW_BYTES + ((chunk ^ (kk * FG::CW)) << 4) + sub;
      }
    }
  }

  acc_t acc[WJ][4];
#pragma unroll
  for (int j = 0; j < WJ; j++)
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int r = 0; r < 16; r++)
        acc[j][i][r] = 0;

  const int64_t b_step = TB ? (int64_t)FG::KB : (int64_t)FG::BK * ldb_b; // bytes from one k-block of B to the next
  // K slice of this workgroup in ring groups (NST stages each): slices differ by at most one group
  const int groups = (int)(p.K / FG::BK) / NST, nsl = SPLIT ? p.splits : 1;
  const int g0 = (int)((int64_t)slice * groups / nsl), g1 = (int)((int64_t)(slice + 1) * groups / nsl);
  const int KT = (g1 - g0) * NST;
  const char *a_ptr = reinterpret_cast<const char *>(p.A) + m0 * lda_b + (int64_t)g0 * NST * FG::KB; // first k-block; KB bytes each
  const char *b_ptr = reinterpret_cast<const char *>(p.B) + (TB ? n0 * ldb_b : n0 * ES) + (int64_t)g0 * NST * b_step;

  uint4 a0[4], b0[WJ], a1[4], b1[WJ];
  // column parameters of this tile: requested before the operand traffic, written to LDS in front of the
  // prologue's barrier (which also publishes them to every wave)
  float cp_bias = -0.0f, cp_scale = 1.0f;
  int cp_cs = 0;
  if constexpr (!SPLIT) {
    if (tid < G_BN) {
      const int64_t n = n0 + tid;
      if (p.bias)
        cp_bias = p.bias_dt == DT_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p.bias)[n])
                                       : reinterpret_cast<const float *>(p.bias)[n];
      if (ES == 1) {
        if (p.scale)
          cp_scale = p.scale[n];
        if (p.colsum)
          cp_cs = p.comp * p.colsum[n];
      }
    }
  }
  // prologue: request k-blocks 0 .. NST-2 (KT is a positive multiple of NST), wait for block 0
#pragma unroll
  for (int d = 0; d < NST - 1; d++)
    g.issue_loads(smem + d * FG::STAGE_BYTES, a_ptr + d * FG::KB, b_ptr + d * b_step);
  if constexpr (!SPLIT) {
    if (tid < G_BN) {
      colp[tid] = cp_bias;
      colp[G_BN + tid] = cp_scale;
      reinterpret_cast<int *>(colp)[2 * G_BN + tid] = cp_cs;
    }
  }
  FG::template wait_dma<NST - 2>();
  __builtin_amdgcn_s_barrier();
  g.load_frags(smem, 0, a0, b0);

  // steady state: groups of NST stages in which every stage still has a block to request
  int kt0 = 0;
  for (; kt0 + 2 * NST <= KT; kt0 += NST) {
    static_for<0, NST>([&](auto sc) {
      constexpr int st = decltype(sc)::value;
      constexpr int cur = st, nxt = (st + 1) % NST, fill = (st + NST - 1) % NST;
      const int kf = kt0 + st + NST - 1;
      g.template stage<true, true, NST - 2>(smem + cur * FG::STAGE_BYTES, smem + nxt * FG::STAGE_BYTES,
                                            smem + fill * FG::STAGE_BYTES, a_ptr + (int64_t)kf * FG::KB,
                                            b_ptr + kf * b_step, acc, a0, b0, a1, b1);
    });
  }
  // last group: only its first stage requests a block (the last one); the ring drains
  static_for<0, NST>([&](auto sc) {
    constexpr int st = decltype(sc)::value;
    constexpr int cur = st, nxt = (st + 1) % NST, fill = (st + NST - 1) % NST;
    constexpr int behind = NST - 2 - st > 0 ? NST - 2 - st : 0;
    const int kf = kt0 + st + NST - 1;
    g.template stage<st == 0, (st < NST - 1), behind>(smem + cur * FG::STAGE_BYTES, smem + nxt * FG::STAGE_BYTES,
                                                      smem + fill * FG::STAGE_BYTES, a_ptr + (int64_t)kf * FG::KB,
                                                      b_ptr + kf * b_step, acc, a0, b0, a1, b1);
  });

  // no wave reads fragments any more (the last stage's barrier came after its
  // final fragment reads), so the stage buffers can be overwritten
  if constexpr (SPLIT) {
    // f32 partial sums of the rows that exist, 16 bytes per lane (4 consecutive n of one m)
    float *part = p.partial + (int64_t)slice * p.M * p.N;
    static_for<0, WJ>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      static_for<0, 4>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const int64_t m = m0 + wm * 128 + i * 32 + l32;
        if (m < p.M) {
#pragma unroll
          for (int q = 0; q < 4; q++) {
            const int64_t n = n0 + wn * (32 * WJ) + j * 32 + 8 * q + 4 * lh;
            f32x4_t v = {(float)acc[j][i][4 * q], (float)acc[j][i][4 * q + 1], (float)acc[j][i][4 * q + 2],
                         (float)acc[j][i][4 * q + 3]};
            *reinterpret_cast<f32x4_t *>(part + m * p.N + n) = v;
          }
        }
      });
    });
    return; // the sum over slices and the epilogue are the second kernel's (a kernel boundary is the cheapest
            // way to make partial sums visible across XCDs: device-scope fences write back and invalidate whole L2s)
  }
  if constexpr (!SPLIT) {
    if (p.out_dt == DT_BF16)
      gemm_epilogue<ES, false, true, WJ, true>(p, acc, m0, n0, wm, wn, l32, lh, smem + wave * (128 * (64 * WJ + 16)), colp);
    else
      gemm_epilogue<ES, false, false, WJ, true>(p, acc, m0, n0, wm, wn, l32, lh, nullptr, colp);
  }
}

// ---------------------------------------------------------------------------
// The whole-tile kernel on v_mfma_f32_16x16x32_bf16 / v_mfma_i32_16x16x64_i8 (B stored [K,N], no K slices).  Same
// tile, ring, DMA and epilogue as gemm_tile256_fast_kernel<ES, 2, 2>; what differs is the MFMA shape.  The board holds a power limit by
// lowering the clock, and per multiply-accumulate the 16x16x32 form moves less register-file data (0.25 B of
// accumulator + 0.25 B of operands against 0.5 B + 0.125 B): a loop of nothing but MFMAs sustains 2.13 PFLOP/s at
// 2.29 GHz with it and 1.89 PFLOP/s at 2.11 GHz with 32x32x16.
// One ring stage (64 bytes of K per row) is exactly one k-step of 32.  A wave's 128 x 64 tile is 8 x 4 tiles of
// 16 x 16; the stage is computed in two halves of 16 MFMAs (row tiles 0-3, then 4-7).  Register fragments: the
// A tiles of the half being computed and of the half to come (2 x 16 registers) and one set of B tiles (16).
// First half: read the A tiles of the second half (and B tile 3).  Barrier (next stage published).  Second half:
// read the next stage's first-half A tiles, and B tiles 0-2 as soon as their last MFMAs of this stage are issued.
#ifndef G_FAST_MI16
#define G_FAST_MI16 1
#endif
#ifndef G_MI16_SPLIT
#define G_MI16_SPLIT 3
#endif
// TB: B stored [N,K]; its tile is staged and read like the A tile (plain 16-byte fragment reads).
template <int ES, bool TB = false> __global__ __launch_bounds__(512, 1) void gemm_tile256_mi16_kernel(GemmParams p) {
  static_assert(!TB || ES == 2, "B stored [N,K]: bf16 only");
  typedef FastGemm<ES, 2, 2, false, TB> FG;
  typedef typename std::conditional<ES == 2, f32x4_t, i32x4_t>::type acc4_t;
  constexpr int NST = FG::NST;
  // one array: the ring / epilogue staging, then the column parameters (see gemm_tile256_fast_kernel)
  __shared__ __align__(1024) char smem[8 * G_STG_WAVE_BYTES + 3 * G_BN * 4];
  float *colp = reinterpret_cast<float *>(smem + 8 * G_STG_WAVE_BYTES);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 2, wn = wave & 3;
  const int l32 = lane & 31, lh = lane >> 5;
  const int r16 = lane & 15, g16 = lane >> 4;

  const int tiles_m = (int)(p.M / G_BM), tiles_n = (int)(p.N / G_BN);
  int tm, tn;
  tile_of_block(blockIdx.x, gridDim.x, tiles_m, tiles_n, p.group_m, tm, tn);
  const int64_t m0 = (int64_t)tm * G_BM, n0 = (int64_t)tn * G_BN;
  const int64_t lda_b = p.lda * ES, ldb_b = p.ldb * ES;
  {
    const int64_t bz = blockIdx.y; // strided batch
    p.A = reinterpret_cast<const char *>(p.A) + bz * p.a_bs * ES;
    p.B = reinterpret_cast<const char *>(p.B) + bz * p.b_bs * ES;
    p.C = reinterpret_cast<char *>(p.C) + bz * p.c_bs * (p.out_dt == DT_BF16 ? 2 : 4);
    if (p.residual)
      p.residual = reinterpret_cast<const char *>(p.residual) + bz * p.c_bs * (p.residual_dt == DT_BF16 ? 2 : 4);
  }

  FG g;
  g.wave_u = wave;
  g.a_xor = p.a_xor;
#pragma unroll
  for (int i = 0; i < FG::NDMA; i++) { // as in gemm_tile256_fast_kernel
    const int row = (wave * FG::NDMA + i) * FG::A_ROWS_PER_DMA + lane / FG::A_CPR;
    const int c = (lane % FG::A_CPR) ^ FG::a_swz(row);
    g.a_src[i] = (uint32_t)(row * lda_b + c * 16);
    const int krow = (wave * FG::NDMA + i) * FG::B_ROWS_PER_DMA + lane / FG::B_CPR;
    const int cb = (lane % FG::B_CPR) ^ ((krow % FG::RG) * FG::CW);
    g.b_src[i] = TB ? (uint32_t)(row * ldb_b + c * 16) : (uint32_t)(krow * ldb_b + cb * 16);
  }
  // A tile `it` (16 rows): lane -> row lane%16, logical 16-byte chunk lane/16 of the row's 64 bytes (8 bf16 or
  // 16 int8 of k)
  const int row_a = wm * 128 + r16; // + 16*it: leaves the swizzle unchanged
  const uint32_t a_ld = (uint32_t)(row_a * FG::KB + ((g16 ^ FG::a_swz(row_a)) << 4));
  // B tile `jt` (16 columns): the 16 lanes of a group hand the transposing read an RG (k) x 16 (n) block of 8-byte
  // pieces (bf16: k row lane%16/4, columns 4*(lane%4)..+3; int8: k row lane%16/2, columns 8*(lane%2)..+7) and get
  // back column lane%16 of those RG k rows; group lane/16 takes k rows 2*RG*(lane/16)..+RG-1 and, 2048 bytes (RG
  // k rows) on, the RG after them
  uint32_t b_ld[4];
  {
    const int kk = ES == 2 ? (r16 >> 2) : (r16 >> 1);
    const int cc = ES == 2 ? (r16 & 3) : (r16 & 1);
#pragma unroll
    for (int jt = 0; jt < 4; jt++) {
      const int chunk = ES == 2 ? (wn * 4 + jt) * 2 + (cc >> 1) : (wn * 4 + jt);
      const int sub = ES == 2 ? (cc & 1) * 8 : cc * 8;
      b_ld[jt] = (uint32_t)(FG::A_BYTES + (2 * FG::RG * g16 + kk) * FG::B_ROW_BYTES + ((chunk ^ (kk * FG::CW)) << 4) + sub);
      if (TB) { // row of the [N,K] tile = column of C; chunk and swizzle as for A
        const int row_b = wn * 64 + jt * 16 + r16;
        b_ld[jt] = (uint32_t)(FG::A_BYTES + row_b * FG::KB + ((g16 ^ FG::a_swz(row_b)) << 4));
      }
    }
  }

  acc4_t acc4[2][4][4]; // [j][i][q]: the 16 x 16 tile at columns 16*(q/2), rows 16*(q%2) of the 32 x 32 block (j, i)
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int q = 0; q < 4; q++)
        acc4[j][i][q] = acc4_t{0, 0, 0, 0};

  const int64_t b_step = TB ? (int64_t)FG::KB : (int64_t)FG::BK * ldb_b;
  const int KT = (int)(p.K / FG::BK); // a positive multiple of NST (checked by the launcher)
  const char *a_ptr = reinterpret_cast<const char *>(p.A) + m0 * lda_b;
  const char *b_ptr = reinterpret_cast<const char *>(p.B) + (TB ? n0 * ldb_b : n0 * ES);

  uint4 a_lo[4], a_hi[4], bb[4];
  auto load_a = [&](const char *__restrict__ st, int half, uint4(&a)[4]) {
#pragma unroll
    for (int ii = 0; ii < 4; ii++) {
      uint4 v = *reinterpret_cast<const uint4 *>(st + a_ld + (half * 4 + ii) * (16 * FG::KB));
      if (ES == 1) // u8 activations: a - 128 as s8 == a ^ 0x80
        v = make_uint4(v.x ^ g.a_xor, v.y ^ g.a_xor, v.z ^ g.a_xor, v.w ^ g.a_xor);
      a[ii] = v;
    }
  };
  auto load_b_tile = [&](const char *__restrict__ st, int jt) -> uint4 {
    if constexpr (TB) {
      return *reinterpret_cast<const uint4 *>(st + b_ld[jt]);
    } else {
      const uint2 lo = MfmaOp<ES>::tr_read(st + b_ld[jt]);
      const uint2 hi = MfmaOp<ES>::tr_read(st + b_ld[jt] + FG::RG * FG::B_ROW_BYTES);
      return make_uint4(lo.x, lo.y, hi.x, hi.y);
    }
  };
  auto load_b = [&](const char *__restrict__ st, uint4(&b)[4]) {
#pragma unroll
    for (int jt = 0; jt < 4; jt++)
      b[jt] = load_b_tile(st, jt);
  };
  // 16 MFMAs: row tiles 4*HALF..+3 against the 4 column tiles; operand roles swapped as in the 32x32 kernels
  // (first operand = B fragment), so a lane ends up with 4 consecutive columns of one row
  auto mfma_half = [&](auto halfc, auto jt0c, auto jt1c, const uint4(&a)[4], const uint4(&b)[4]) {
    constexpr int HALF = decltype(halfc)::value, JT0 = decltype(jt0c)::value, JT1 = decltype(jt1c)::value;
    static_for<JT0, JT1>([&](auto jtc) {
      constexpr int jt = decltype(jtc)::value;
      static_for<0, 4>([&](auto iic) {
        constexpr int it = HALF * 4 + decltype(iic)::value;
        constexpr int j = jt >> 1, i = it >> 1, q = 2 * (jt & 1) + (it & 1);
        if constexpr (ES == 2)
          acc4[j][i][q] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, b[jt]),
                                                                  __builtin_bit_cast(bf16x8_t, a[it & 3]), acc4[j][i][q], 0, 0, 0);
        else
          acc4[j][i][q] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, b[jt]),
                                                                __builtin_bit_cast(i32x4_t, a[it & 3]), acc4[j][i][q], 0, 0, 0);
      });
    });
  };
  // MFMA, two LDS reads, MFMA, two LDS reads ... until the group's reads are out, then the remaining MFMAs
  auto hint = [&](auto ndsc, auto nmc) {
    constexpr int N_DS = decltype(ndsc)::value, N_MFMA = decltype(nmc)::value;
    static_for<0, N_MFMA>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      constexpr int left = N_DS - 2 * i;
      if constexpr (left > 0)
        __builtin_amdgcn_sched_group_barrier(0x100, left < 2 ? left : 2, 0);
    });
  };
  // One stage (see FastGemm::stage for the ring).  MFMAs run column tile by column tile; a column tile's B fragment
  // is dead after its four MFMAs of the second half and is reloaded from the next stage on the spot, so B needs one
  // set of registers.
  auto stage = [&](auto has_fill, auto has_next, auto behindc, char *__restrict__ cur, char *__restrict__ nxt,
                   char *__restrict__ fill, const char *a_fill, const char *b_fill) {
    constexpr bool HAS_FILL = decltype(has_fill)::value, HAS_NEXT = decltype(has_next)::value;
    constexpr int BEHIND = decltype(behindc)::value;
    typedef std::integral_constant<int, 0> I0;
    typedef std::integral_constant<int, 1> I1;
    typedef std::integral_constant<int, G_MI16_SPLIT> I3; // column tiles of the first half in front of the barrier
    typedef std::integral_constant<int, 4> I4;
    if constexpr (HAS_FILL)
      g.issue_loads(fill, a_fill, b_fill);
    load_a(cur, 1, a_hi);
    // the last column tile's B fragment is first read behind the barrier: fetched here rather than at the very end
    // of the previous stage, where the (full) LDS wait in front of this half would have to sit it out
    bb[3] = load_b_tile(cur, 3);
    mfma_half(I0{}, I0{}, I3{}, a_lo, bb); // 12 of the first half's 16
    hint(std::integral_constant<int, TB ? 5 : 6>{}, std::integral_constant<int, 4 * G_MI16_SPLIT>{});
    // The barrier sits three quarters into the first half: the reads above have returned by then (its wait covers
    // them), and the four MFMAs left over cover the barrier's own latency.  Nothing may move across it.
    __builtin_amdgcn_sched_barrier(0);
    FG::template wait_dma<BEHIND>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    mfma_half(I0{}, I3{}, I4{}, a_lo, bb); // the last readers of a_lo
    if constexpr (HAS_NEXT)
      load_a(nxt, 0, a_lo);
    static_for<0, 4>([&](auto jtc) {
      constexpr int jt = decltype(jtc)::value;
      mfma_half(I1{}, jtc, std::integral_constant<int, jt + 1>{}, a_hi, bb);
      if constexpr (HAS_NEXT && jt < 3)
        bb[jt] = load_b_tile(nxt, jt);
    });
    // issue order after the barrier: the four MFMAs left of the first half; the next stage's first-half A tiles
    // between the MFMAs of column tile 0; after each column tile its B fragment of the next stage
    if constexpr (G_MI16_SPLIT < 4)
      __builtin_amdgcn_sched_group_barrier(0x008, 4 * (4 - G_MI16_SPLIT), 0);
    static_for<0, 4>([&](auto ic) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      if constexpr (HAS_NEXT)
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
    });
    static_for<0, 4>([&](auto jtc) {
      if constexpr (decltype(jtc)::value > 0)
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
      if constexpr (HAS_NEXT && decltype(jtc)::value < 3)
        __builtin_amdgcn_sched_group_barrier(0x100, TB ? 1 : 2, 0);
    });
  };

  // column parameters of this tile (see gemm_tile256_fast_kernel)
  float cp_bias = -0.0f, cp_scale = 1.0f;
  int cp_cs = 0;
  if (tid < G_BN) {
    if (p.bias)
      cp_bias = p.bias_dt == DT_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p.bias)[n0 + tid])
                                     : reinterpret_cast<const float *>(p.bias)[n0 + tid];
    if (ES == 1) {
      if (p.scale)
        cp_scale = p.scale[n0 + tid];
      if (p.colsum)
        cp_cs = p.comp * p.colsum[n0 + tid];
    }
  }
#pragma unroll
  for (int d = 0; d < NST - 1; d++)
    g.issue_loads(smem + d * FG::STAGE_BYTES, a_ptr + d * FG::KB, b_ptr + d * b_step);
  if (tid < G_BN) {
    colp[tid] = cp_bias;
    colp[G_BN + tid] = cp_scale;
    reinterpret_cast<int *>(colp)[2 * G_BN + tid] = cp_cs;
  }
  FG::template wait_dma<NST - 2>();
  __builtin_amdgcn_s_barrier();
  load_a(smem, 0, a_lo);
  load_b(smem, bb);

  typedef std::integral_constant<bool, true> T;
  typedef std::integral_constant<bool, false> F;
  int kt0 = 0;
  for (; kt0 + 2 * NST <= KT; kt0 += NST) {
    static_for<0, NST>([&](auto sc) {
      constexpr int st = decltype(sc)::value;
      constexpr int cur = st, nxt = (st + 1) % NST, fill = (st + NST - 1) % NST;
      const int kf = kt0 + st + NST - 1;
      stage(T{}, T{}, std::integral_constant<int, NST - 2>{}, smem + cur * FG::STAGE_BYTES, smem + nxt * FG::STAGE_BYTES, smem + fill * FG::STAGE_BYTES,
            a_ptr + (int64_t)kf * FG::KB, b_ptr + kf * b_step);
    });
  }
  static_for<0, NST>([&](auto sc) { // last group: only its first stage requests a block; the ring drains
    constexpr int st = decltype(sc)::value;
    constexpr int cur = st, nxt = (st + 1) % NST, fill = (st + NST - 1) % NST;
    constexpr int behind = NST - 2 - st > 0 ? NST - 2 - st : 0;
    const int kf = kt0 + st + NST - 1;
    stage(std::integral_constant<bool, st == 0>{}, std::integral_constant<bool, (st < NST - 1)>{},
          std::integral_constant<int, behind>{}, smem + cur * FG::STAGE_BYTES,
          smem + nxt * FG::STAGE_BYTES, smem + fill * FG::STAGE_BYTES, a_ptr + (int64_t)kf * FG::KB, b_ptr + kf * b_step);
  });

  // the accumulators in the shape the epilogue takes: element 4q+e of block (j, i)
  typename MfmaOp<ES>::acc_t acc[2][4];
#pragma unroll
  for (int j = 0; j < 2; j++)
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int q = 0; q < 4; q++)
#pragma unroll
        for (int e = 0; e < 4; e++)
          acc[j][i][4 * q + e] = acc4[j][i][q][e];
  if (p.out_dt == DT_BF16)
    gemm_epilogue<ES, false, true, 2, true, true>(p, acc, m0, n0, wm, wn, l32, lh, smem + wave * G_STG_WAVE_BYTES, colp);
  else
    gemm_epilogue<ES, false, false, 2, true, true>(p, acc, m0, n0, wm, wn, l32, lh, nullptr, colp);
}

// ---------------------------------------------------------------------------
// The kernels with one wave per SIMD and a hand-placed main loop: 4 waves as 2 x 2, each owning MI x NJ tiles of 16 x 16
// (v_mfma_f32_16x16x32_bf16 / v_mfma_i32_16x16x64_i8).  8 x 8: the 256 x 256 tile, 256 accumulator registers; against
// the 8-wave kernel a multiply-accumulate costs a third less LDS read traffic (per k-step a wave reads 8 KiB of A
// and 8 KiB of B for 64 MFMAs, not 8 + 4 KiB for 32), which is what counts on a board that holds its power limit
// by lowering the clock.  8 x 4 and 6 x 4: 256 and 192 rows by 128 columns, for problems that large tiles leave half the GPU idle.
// With a single wave per SIMD nothing hides a stall, so every fragment is fetched a whole
// stage ahead: stage t computes k-block t from registers, and between its MFMAs the wave reads k-block t+1 into the other
// register set and requests what the LDS ring has room for, two to four stages ahead.  Operands whose rows run along K are
// requested in pairs of k-blocks, 128 bytes of a row at a time (whole cache lines), B stored [K,N] block by block.
// Against requests of single k-blocks (half lines, each line fetched from L2 twice: the line reads of L2 are what large tiles
// then wait for) and, for the 128-column tiles, against a loop left to the compiler, us, weights [K,N] / [N,K], from memory:
// 4096^3 99.3 -> 96.6 / 116 -> 94.5; 1000 x 11008, K 4096 (with its 172 tiles dealt to the XCDs in runs) 92 -> 78 / 118 -> 81;
// 1000 x 4096, K 11008 (256 x 128, two slices) 117 -> 94 / 121 -> 97; 1237 x 4096, K 1376 (192 x 128) 26.4 -> 23.8 / 28.4 -> 25.8;
// 8-bit 4096 x 4096 x 11008 with its epilogue 158.3 -> 155.8.
// The main loop is assembly text written by gen_gemm_w4_mainloop.py, which has the details (registers and issue order fixed
// by hand: the compiler's allocator does not hold 64 accumulator tiles and four fragment sets without copies and spills);
// set-up and epilogue are the C++ below.
#include "gemm_w4_mainloop.inc"

// Epilogue of gemm_tile256_w4_kernel.  The main loop's assembly ends by writing the raw accumulators of column
// tiles 0-3 (the left 64 columns of the wave's 128 x 128) to a wave-private LDS region, 128 rows of 256 bytes at a
// pitch of 272; a second, small assembly statement does the same for column tiles 4-7 once the first half has been
// consumed.  What is left for this code is a rolled loop over rows: a lane reads four consecutive columns of a row
// (16 bytes, 16 lanes per row, 4 rows per instruction), applies the epilogue and stores 8 (bf16) or 16 bytes, so a
// row leaves as one or two whole 128-byte lines.  Unrolled over the 64 accumulator tiles in place of the loop, the
// same work was ten times the code, all of it executed once per workgroup and fetched cold: 12 us of a 100 us
// kernel went into instruction-cache misses.
static constexpr int W4_DUMP_PITCH = 272;                   // 64 f32 / s32 + 16 bytes: conflict-free for the 16-byte writes

// Four results of one row: c = the raw accumulators of columns n .. n+3 of row m.  HAS_BIAS / HAS_RES are
// compile-time so that the eight rows of an unrolled group are straight-line code (their LDS reads go out together).
// NAN_FREE: the caller has shown that no result of this row can be a NaN, so the bf16 conversions need no fix-up.
// MASKED (a tile that sticks out of C): row_ok says whether row m exists; nothing of a missing row is read or stored.
template <int ES, int ACT, int OUT, bool HAS_BIAS, bool HAS_RES, bool MASKED, bool NAN_FREE = false, typename acc4_t>
__device__ __forceinline__ void w4_epilogue_row(const GemmParams &p, const acc4_t &c, int64_t m, int64_t n,
                                                const f32x4_t &bias4, const f32x4_t &scale4, const i32x4_t &cs4,
                                                bool row_ok = true) {
  if (MASKED && !row_ok)
    return;
  char *Cb = reinterpret_cast<char *>(p.C);
  float x[4];
  uint32_t p0 = 0, p1 = 0; // bf16 results, two per register
  if constexpr (ES == 1) {
    int ci[4];
#pragma unroll
    for (int e = 0; e < 4; e++)
      ci[e] = (int)c[e] + cs4[e]; // exact: the zero-point term in integer arithmetic
    if constexpr (OUT == DT_S32) {
      *reinterpret_cast<i32x4_t *>(Cb + (m * p.ldc + n) * 4) = i32x4_t{ci[0], ci[1], ci[2], ci[3]};
      return;
    }
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const float v = fmaf((float)ci[e], scale4[e], bias4[e]); // an absent bias is -0.0: the product itself
#ifndef GCMI_GELU_BF16_PRECISE // (measurement builds define it to time the f32-grade erf in this place)
      if constexpr (OUT == DT_BF16 && NAN_FREE && ACT == ACT_GELU_ERF)
        x[e] = gelu_erf_bf16_result(v); // v is finite here and the result is rounded to bf16 below
      else
#endif
        x[e] = act_const<ACT>(v);
    }
    if constexpr (OUT == DT_F32) {
      *reinterpret_cast<f32x4_t *>(Cb + (m * p.ldc + n) * 4) = f32x4_t{x[0], x[1], x[2], x[3]};
      return;
    }
    // v_cvt_pk_bf16_f32 rounds to nearest even but keeps a NaN's sign and payload; a NaN among the four (their
    // sum is one; so is the sum of opposite infinities) sends them through the scalar rule: NaN -> 0x7FC0
    const float any_nan = NAN_FREE ? 0.0f : (x[0] + x[1]) + (x[2] + x[3]);
    if (__builtin_expect(any_nan != any_nan, 0)) {
      p0 = f32_to_bf16_bits(x[0]) | ((uint32_t)f32_to_bf16_bits(x[1]) << 16);
      p1 = f32_to_bf16_bits(x[2]) | ((uint32_t)f32_to_bf16_bits(x[3]) << 16);
    } else {
      p0 = pack_bf16x2(x[0], x[1]), p1 = pack_bf16x2(x[2], x[3]);
    }
  } else {
#pragma unroll
    for (int e = 0; e < 4; e++)
      x[e] = (float)c[e];
    float res4[4] = {0.f, 0.f, 0.f, 0.f};
    if constexpr (HAS_RES) { // 16-byte aligned rows (checked by the launcher)
      const int64_t at = m * p.ldr + n;
      if (p.residual_dt == DT_BF16) {
        const uint2 v = *reinterpret_cast<const uint2 *>(reinterpret_cast<const uint16_t *>(p.residual) + at);
        res4[0] = __uint_as_float(v.x << 16), res4[1] = __uint_as_float(v.x & 0xffff0000u);
        res4[2] = __uint_as_float(v.y << 16), res4[3] = __uint_as_float(v.y & 0xffff0000u);
      } else {
        const f32x4_t v = *reinterpret_cast<const f32x4_t *>(reinterpret_cast<const float *>(p.residual) + at);
        res4[0] = v[0], res4[1] = v[1], res4[2] = v[2], res4[3] = v[3];
      }
    }
    if constexpr (OUT == DT_F32) { // no intermediate rounding
#pragma unroll
      for (int e = 0; e < 4; e++) {
        if constexpr (HAS_BIAS)
          x[e] = x[e] + bias4[e];
        x[e] = act_const<ACT>(x[e]);
        if constexpr (HAS_RES) { // kept apart from the activation's last multiply: the sum equals a separate add
#pragma clang fp contract(off)
          x[e] = x[e] + res4[e];
        }
      }
      *reinterpret_cast<f32x4_t *>(Cb + (m * p.ldc + n) * 4) = f32x4_t{x[0], x[1], x[2], x[3]};
      return;
    }
    // bf16 graph: rounded after the matmul and after every bf16 op (lib/gc/Transforms/Pipeline.cpp:79-95), in
    // pairs.  A NaN stays a NaN through the ops that follow, so only the last conversion gives it 0x7FC0.
    auto rnd = [&]() {
      p0 = pack_bf16x2(x[0], x[1]), p1 = pack_bf16x2(x[2], x[3]);
      x[0] = __uint_as_float(p0 << 16), x[1] = __uint_as_float(p0 & 0xffff0000u);
      x[2] = __uint_as_float(p1 << 16), x[3] = __uint_as_float(p1 & 0xffff0000u);
    };
    constexpr bool LAST_IS_MATMUL = !HAS_BIAS && ACT == ACT_NONE && !HAS_RES;
    if constexpr (LAST_IS_MATMUL) { // nothing follows the first rounding: no need to widen again
      p0 = pack_bf16x2(x[0], x[1]), p1 = pack_bf16x2(x[2], x[3]);
    } else {
      rnd();
    }
    if constexpr (HAS_BIAS) {
#pragma unroll
      for (int e = 0; e < 4; e++)
        x[e] = x[e] + bias4[e];
      rnd();
    }
    if constexpr (ACT != ACT_NONE) {
#pragma unroll
      for (int e = 0; e < 4; e++) // (GELU by erf / so, us: 1237 x 4096, K 1376 23.4 / 22.2; 2048 x 8192, K 512 29.3 / 25.6)
        x[e] = apply_act_of_bf16(x[e], ACT);
      if constexpr (ACT == ACT_RELU) { // max(x, 0) of a bf16 value is a bf16 value: nothing to round
        p0 = (__float_as_uint(x[0]) >> 16) | (__float_as_uint(x[1]) & 0xffff0000u);
        p1 = (__float_as_uint(x[2]) >> 16) | (__float_as_uint(x[3]) & 0xffff0000u);
      } else {
        rnd();
      }
    }
    if constexpr (HAS_RES) {
#pragma unroll
      for (int e = 0; e < 4; e++)
        x[e] = x[e] + res4[e];
      rnd();
    }
    const float any_nan = NAN_FREE ? 0.0f : (x[0] + x[1]) + (x[2] + x[3]);
    if (__builtin_expect(any_nan != any_nan, 0)) {
      if (x[0] != x[0]) p0 = (p0 & 0xffff0000u) | 0x7FC0u;
      if (x[1] != x[1]) p0 = (p0 & 0x0000ffffu) | 0x7FC00000u;
      if (x[2] != x[2]) p1 = (p1 & 0xffff0000u) | 0x7FC0u;
      if (x[3] != x[3]) p1 = (p1 & 0x0000ffffu) | 0x7FC00000u;
    }
  }
  typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
  const u32x2_t vv = {p0, p1};
  __builtin_nontemporal_store(vv, reinterpret_cast<u32x2_t *>(Cb + (m * p.ldc + n) * 2));
}

// One half (64 columns) of the wave tile.  OUT = DT_BF16 / DT_F32 / DT_S32.
// MASKED: rows_in / cols_in of the tile's 256 x 256 lie inside C (cols_in is a multiple of 4).
// WR x WC: the wave's tile (128 x 128 in the 256 x 256 kernel, 64 x 64 in the 128 x 128 one); rows_in / cols_in count
// from the workgroup tile's corner whatever its size.
template <int ES, int ACT, int OUT, bool MASKED, int WR = 128, int WC = 128>
__device__ __forceinline__ void w4_epilogue_half(const GemmParams &p, int half, int64_t m0, int64_t n0, int wm, int wn,
                                                 int lane, const char *dump, const float *colp, int rows_in, int cols_in) {
  typedef typename std::conditional<ES == 2, float, int>::type acc_e;
  typedef acc_e acc4_t __attribute__((ext_vector_type(4)));
  const int rr = lane >> 4, cc = lane & 15;
  const int col = wn * WC + half * 64 + 4 * cc; // this lane's four columns inside the workgroup tile
  const int64_t n = n0 + col;
  if (MASKED && col >= cols_in)
    return;
  if (WC % 64 != 0 && half * 64 + 4 * cc >= WC) // the last 32 columns of a wave tile of 96
    return;
  const int row0 = wm * WR + rr; // + 4 * (i0 + u)
  const f32x4_t bias4 = *reinterpret_cast<const f32x4_t *>(colp + col); // -0.0 where there is no bias
  f32x4_t scale4 = {1.f, 1.f, 1.f, 1.f};
  i32x4_t cs4 = {0, 0, 0, 0}; // comp * colsum
  if constexpr (ES == 1) {
    scale4 = *reinterpret_cast<const f32x4_t *>(colp + 256 + col);
    cs4 = *reinterpret_cast<const i32x4_t *>(colp + 512 + col);
  }
  const bool has_bias = ES == 2 && p.bias != nullptr, has_res = ES == 2 && p.residual != nullptr;
  const bool bias_finite = fabsf((bias4[0] + bias4[1]) + (bias4[2] + bias4[3])) < __builtin_inff() || // the usual case
                           (fabsf(bias4[0]) < __builtin_inff() && fabsf(bias4[1]) < __builtin_inff() &&
                            fabsf(bias4[2]) < __builtin_inff() && fabsf(bias4[3]) < __builtin_inff());
  const bool bias_tame = fabsf(bias4[0]) < 0x1p120f && fabsf(bias4[1]) < 0x1p120f && fabsf(bias4[2]) < 0x1p120f && fabsf(bias4[3]) < 0x1p120f;
  bool cols_tame = true;
  if constexpr (ES == 1) {
#pragma unroll
    for (int e = 0; e < 4; e++)
      cols_tame = cols_tame && fabsf(scale4[e]) < 0x1p90f && fabsf(bias4[e]) < 0x1p120f;
  }
  constexpr int U = 8; // rows in flight per lane
#pragma unroll 1
  for (int i0 = 0; i0 < WR / 4; i0 += U) {
    // none of the wave's 4 * U rows from here on lies inside (passed over: 3 x 2312, K 96 with GELU 13.3 us -> 9.9; 2 x 1192, K 136 14.6 -> 11.4).
    // Waves of 64 rows have two groups and only pay for the question: 8-bit 63 x 544, K 64 with GELU 6.95 us -> 7.1, 1437 x 976, K 112 7.15 -> 7.28
    if (MASKED && WR > 64 && wm * WR + 4 * i0 >= rows_in)
      return;
    acc4_t c[U];
#pragma unroll
    for (int u = 0; u < U; u++)
      c[u] = *reinterpret_cast<const acc4_t *>(dump + ((i0 + u) * 4 + rr) * W4_DUMP_PITCH + cc * 16);
    auto rows = [&](auto hb, auto hr) {
      constexpr bool HB = decltype(hb)::value, HR = decltype(hr)::value;
      // bf16 results of finite accumulators and finite biases through nothing but an add and a ReLU are no NaNs:
      // one sum over the group's 32 accumulators (a NaN or an infinity among them makes it non-finite) replaces
      // the check of every row
      if constexpr (ES == 2 && OUT == DT_BF16 && !HR && (ACT == ACT_NONE || ACT == ACT_RELU)) {
        float t = 0.0f;
#pragma unroll
        for (int u = 0; u < U; u++)
          t += ((float)c[u][0] + (float)c[u][1]) + ((float)c[u][2] + (float)c[u][3]);
        if (__builtin_expect(bias_finite && fabsf(t) < __builtin_inff(), 1)) {
#pragma unroll
          for (int u = 0; u < U; u++)
            w4_epilogue_row<ES, ACT, OUT, HB, HR, MASKED, true>(p, c[u], m0 + row0 + (i0 + u) * 4, n, bias4, scale4, cs4,
                                                                row0 + (i0 + u) * 4 < rows_in);
          return;
        }
      }
      // GELU: a sum of magnitudes, since it makes a NaN of -inf
      if constexpr (ES == 2 && OUT == DT_BF16 && !HR && ACT == ACT_GELU_ERF) {
        float t = 0.0f;
#pragma unroll
        for (int u = 0; u < U; u++)
          t += (fabsf((float)c[u][0]) + fabsf((float)c[u][1])) + (fabsf((float)c[u][2]) + fabsf((float)c[u][3]));
        if (__builtin_expect(bias_tame && t < 0x1p120f, 1)) {
#pragma unroll
          for (int u = 0; u < U; u++)
            w4_epilogue_row<ES, ACT, OUT, HB, HR, MASKED, true>(p, c[u], m0 + row0 + (i0 + u) * 4, n, bias4, scale4, cs4,
                                                                row0 + (i0 + u) * 4 < rows_in);
          return;
        }
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        w4_epilogue_row<ES, ACT, OUT, HB, HR, MASKED>(p, c[u], m0 + row0 + (i0 + u) * 4, n, bias4, scale4, cs4,
                                                      row0 + (i0 + u) * 4 < rows_in);
    };
    typedef std::integral_constant<bool, true> T;
    typedef std::integral_constant<bool, false> F;
    if constexpr (ES == 1) {
      // |acc| < 2^31: with scales below 2^90 and biases below 2^120 in magnitude the dequantised value is finite, and
      // so is every activation of it: no NaN to look for
      if (__builtin_expect(cols_tame, 1)) {
#pragma unroll
        for (int u = 0; u < U; u++)
          w4_epilogue_row<ES, ACT, OUT, false, false, MASKED, true>(p, c[u], m0 + row0 + (i0 + u) * 4, n, bias4, scale4, cs4,
                                                                    row0 + (i0 + u) * 4 < rows_in);
      } else {
        rows(F{}, F{});
      }
    } else {
      if (has_bias) {
        if (has_res)
          rows(T{}, T{});
        else
          rows(T{}, F{});
      } else {
        if (has_res)
          rows(F{}, T{});
        else
          rows(F{}, F{});
      }
    }
  }
}

// kind = act + 8 * (0: bf16, 1: f32, 2: s32)
template <int ES, bool MASKED, int WR = 128, int WC = 128>
__device__ __forceinline__ void w4_epilogue_half_any(const GemmParams &p, int kind, int half, int64_t m0, int64_t n0,
                                                     int wm, int wn, int lane, const char *dump, const float *colp,
                                                     int rows_in, int cols_in) {
#define GCMI_W4_CASE(ACT, OUT, K)                                                                                     \
  case (int)ACT + 8 * K:                                                                                              \
    w4_epilogue_half<ES, ACT, OUT, MASKED, WR, WC>(p, half, m0, n0, wm, wn, lane, dump, colp, rows_in, cols_in);      \
    break;
  switch (kind) {
    GCMI_W4_CASE(ACT_RELU, DT_BF16, 0)
    GCMI_W4_CASE(ACT_GELU_ERF, DT_BF16, 0)
    GCMI_W4_CASE(ACT_GELU_TANH, DT_BF16, 0)
    GCMI_W4_CASE(ACT_SIGMOID, DT_BF16, 0)
    GCMI_W4_CASE(ACT_NONE, DT_F32, 1)
    GCMI_W4_CASE(ACT_RELU, DT_F32, 1)
    GCMI_W4_CASE(ACT_GELU_ERF, DT_F32, 1)
    GCMI_W4_CASE(ACT_GELU_TANH, DT_F32, 1)
    GCMI_W4_CASE(ACT_SIGMOID, DT_F32, 1)
    GCMI_W4_CASE(ACT_NONE, DT_S32, 2)
  default:
    w4_epilogue_half<ES, ACT_NONE, DT_BF16, MASKED, WR, WC>(p, half, m0, n0, wm, wn, lane, dump, colp, rows_in, cols_in);
    break;
  }
#undef GCMI_W4_CASE
}

// 1 / (1 + exp(-x)) of a bf16 value x for a bf16 result: the hardware's exponential and reciprocal, each good to an ulp of f32
// or two, in place of expf and a correctly rounded division (20 issue slots fewer per result).  The sum is a quarter of the true
// one: the reciprocal makes a result below the smallest normal number 0, which is then just where expf(-x) is infinite (2^128
// and more, x = -89 and below).  Rounded to bf16 it is what those give for every bf16 x.
__device__ __forceinline__ float sigmoid_of_bf16(float x) {
  return 0.25f * __builtin_amdgcn_rcpf(0.25f + __builtin_amdgcn_exp2f(fmaf(x, -1.4426950408889634f, -2.0f)));
}

// What a gated pair of products ends in, silu(gate) * up, for four results of a row: both sums rounded to bf16, then the
// graph's three ops (x / (1 + exp(-x)) as sigmoid and product, the product with up), each rounded as a bf16 tensor would
// be.  A NaN stays a NaN through the ops, so only the last conversion gives it 0x7FC0.
__device__ __forceinline__ uint2 gated_silu4(const f32x4_t &gate, const f32x4_t &up) {
  auto rnd = [](float(&x)[4]) {
    const uint32_t a = pack_bf16x2(x[0], x[1]), b = pack_bf16x2(x[2], x[3]);
    x[0] = __uint_as_float(a << 16), x[1] = __uint_as_float(a & 0xffff0000u);
    x[2] = __uint_as_float(b << 16), x[3] = __uint_as_float(b & 0xffff0000u);
  };
  float g[4] = {gate[0], gate[1], gate[2], gate[3]}, u[4] = {up[0], up[1], up[2], up[3]}, x[4];
  rnd(g), rnd(u);
#pragma unroll
  for (int e = 0; e < 4; e++)
    x[e] = sigmoid_of_bf16(g[e]);
  rnd(x);
#pragma unroll
  for (int e = 0; e < 4; e++)
    x[e] = x[e] * g[e];
  rnd(x);
#pragma unroll
  for (int e = 0; e < 4; e++)
    x[e] = x[e] * u[e];
  uint32_t p0 = pack_bf16x2(x[0], x[1]), p1 = pack_bf16x2(x[2], x[3]);
  const float any_nan = (x[0] + x[1]) + (x[2] + x[3]);
  if (__builtin_expect(any_nan != any_nan, 0)) {
    p0 = f32_to_bf16_bits(x[0]) | ((uint32_t)f32_to_bf16_bits(x[1]) << 16);
    p1 = f32_to_bf16_bits(x[2]) | ((uint32_t)f32_to_bf16_bits(x[3]) << 16);
  }
  return make_uint2(p0, p1);
}

// Epilogue of a gated tile: the left wave column holds the gate's sums, the right one those of up, for the same rows and
// columns of C.  Each of the two waves of a wave row takes every other group of four rows of both their regions, up to 64 columns at a time.
template <int WR, int WC>
__device__ __forceinline__ void w4_gated_half(const GemmParams &p, int half, int64_t m0, int64_t n0, int wm, int wn, int lane,
                                              const char *gate, const char *up, int rows_in, int cols_in) {
  const int rr = lane >> 4, cc = lane & 15, col = half * 64 + 4 * cc; // this lane's four columns of C, from n0 on
  if (col >= cols_in || (WC % 64 != 0 && col >= WC))
    return;
  constexpr int U = 4; // rows in flight per lane
#pragma unroll 1
  for (int i0 = wn; i0 < WR / 4; i0 += 2 * U) {
    f32x4_t g[U], v[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int at = ((i0 + 2 * u) * 4 + rr) * W4_DUMP_PITCH + cc * 16;
      g[u] = *reinterpret_cast<const f32x4_t *>(gate + at);
      v[u] = *reinterpret_cast<const f32x4_t *>(up + at);
    }
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int row = wm * WR + (i0 + 2 * u) * 4 + rr;
      if (row >= rows_in)
        continue;
      typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
      const uint2 o = gated_silu4(g[u], v[u]);
      __builtin_nontemporal_store(u32x2_t{o.x, o.y}, reinterpret_cast<u32x2_t *>(reinterpret_cast<uint16_t *>(p.C) +
                                                                                 (m0 + row) * p.ldc + n0 + col));
    }
  }
}

// K not a whole number of ring groups (four k-blocks of 64 bytes): the incomplete group [k_full, K) is the FIRST one
// computed, and this puts it into the ring's four slots before the main loop starts: whole k-blocks by DMA, the block
// that K ends in through registers with zeros behind K (in both operands, so no product of theirs counts, whatever the
// memory behind K holds), zero blocks without a load.  The main loop then requests from k = 0 on; its steady state
// knows nothing of the tail.
// Before, every K that is no multiple of 128 bf16 / 256 bytes went to the bounds-checked kernel: 1237 x 4096 x 1376
// ([N,K] weights) took 89.7 us there, 29.5 us as 320 tiles of 128 x 128.
// a_src / b_src: the lane's byte offset per DMA instruction (NA and NB of them per wave and block); a_k / b_k: its first k inside a block, which decides whether
// it lies before K.
template <int ES, bool TB, int NA, int NB, int STAGE, int A_BYTES, typename OffA, typename OffB>
__device__ __forceinline__ void fill_ring_k_tail(char *smem, int wave, int lane, const char *a_tail, const char *b_tail,
                                                 int64_t b_step, int k_left, const OffA &a_src, const OffB &b_src,
                                                 const int (&a_k)[NA], const int (&b_k)[NB]) {
  constexpr int BK = 64 / ES;
#pragma unroll 1
  for (int blk = 0; blk < 4; blk++, k_left -= BK, a_tail += 64, b_tail += b_step) {
    char *sa = smem + blk * STAGE + wave * NA * 1024, *sb = smem + blk * STAGE + A_BYTES + wave * NB * 1024;
    if (k_left >= BK) {
#pragma unroll
      for (int i = 0; i < NA; i++)
        __builtin_amdgcn_global_load_lds((GCMI_GLB const void *)(a_tail + (uint32_t)a_src[i]), (GCMI_LDS void *)(sa + i * 1024), 16, 0, 0);
#pragma unroll
      for (int i = 0; i < NB; i++)
        __builtin_amdgcn_global_load_lds((GCMI_GLB const void *)(b_tail + (uint32_t)b_src[i]), (GCMI_LDS void *)(sb + i * 1024), 16, 0, 0);
      continue;
    }
    uint4 va[NA], vb[NB];
#pragma unroll
    for (int i = 0; i < NA; i++) {
      va[i] = make_uint4(0, 0, 0, 0);
      if (a_k[i] < k_left)
        va[i] = *reinterpret_cast<const uint4 *>(a_tail + (uint32_t)a_src[i]);
    }
#pragma unroll
    for (int i = 0; i < NB; i++) {
      vb[i] = make_uint4(0, 0, 0, 0);
      if (b_k[i] < k_left)
        vb[i] = *reinterpret_cast<const uint4 *>(b_tail + (uint32_t)b_src[i]);
    }
#pragma unroll
    for (int i = 0; i < NA; i++)
      *reinterpret_cast<uint4 *>(sa + i * 1024 + lane * 16) = va[i];
#pragma unroll
    for (int i = 0; i < NB; i++)
      *reinterpret_cast<uint4 *>(sb + i * 1024 + lane * 16) = vb[i];
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
}

// One operand's zeros / requests of a pair or block of `whole` k, `left` of which lie before K; k: the first k of the lane's 16 bytes.
template <int N> __device__ __forceinline__ void k_tail_zeros(char *to, int lane, const int (&k)[N], int whole, int left) {
  if (left >= whole)
    return;
#pragma unroll
  for (int i = 0; i < N; i++)
    if (k[i] >= left)
      *reinterpret_cast<uint4 *>(to + i * 1024 + lane * 16) = make_uint4(0, 0, 0, 0);
}
template <int N>
__device__ __forceinline__ void k_tail_requests(char *to, const char *from, const int (&off)[8], const int (&k)[N], int whole, int left) {
  auto request = [&](int i) {
    __builtin_amdgcn_global_load_lds((GCMI_GLB const void *)(from + (uint32_t)off[i]), (GCMI_LDS void *)(to + i * 1024), 16, 0, 0);
  };
  if (left <= 0)
    return;
  if (left >= whole) {
#pragma unroll
    for (int i = 0; i < N; i++)
      request(i);
    return;
  }
#pragma unroll
  for (int i = 0; i < N; i++)
    if (k[i] < left)
      request(i);
}
// K not a whole number of groups (two pairs of k-blocks, 256 bytes): the incomplete group [k_full, K) is the FIRST one
// computed, and this puts it into slots 0 and 1 of the rings before the main loop's own requests go out: chunks before K by DMA,
// zeros behind it (in both operands, so no product of theirs counts, whatever the memory behind K holds) by the lanes whose
// chunks those are, which take no part in that request.  Nothing is waited for here: the main loop waits for these requests, the
// oldest, when the next ones are on their way and its accumulators are cleared.  (The pair that K ends in used to go through registers, behind the next requests,
// and everything in flight was waited for: 852 x 1728, K 1104 of 8 bits 11.05 -> 10.37 us, 1796 x 192, K 1176 13.3 -> 12.6,
// 3106 x 3840, K 280 18.5 -> 17.7; 37 random sizes with such a K 1.023 times, none slower.)
template <int ES, bool TB, int MI, int NJ>
__device__ __forceinline__ void w4_request_k_tail(char *smem, int wave, int lane, const char *a_tail, const char *b_tail, int64_t b_step,
                                                  int k_left, const int (&a_off)[8], const int (&b_off)[8], const int (&a_k)[MI],
                                                  const int (&b_k)[TB ? NJ : NJ / 2]) {
  constexpr int BK = 64 / ES, A_PAIR = MI * 4096, B_PAIR = NJ * 4096, NB = TB ? NJ : NJ / 2;
  char *const sa = smem + wave * MI * 1024, *const sb = smem + W4Ring<ES, TB, MI, NJ>::DA * A_PAIR + wave * NB * 1024;
#pragma unroll 1
  for (int q = 0; q < 2; q++) {
    k_tail_zeros<MI>(sa + q * A_PAIR, lane, a_k, 2 * BK, k_left - q * 2 * BK);
#pragma unroll
    for (int h = 0; h < (TB ? 1 : 2); h++)
      k_tail_zeros<NB>(sb + q * B_PAIR + h * (B_PAIR / 2), lane, b_k, TB ? 2 * BK : BK, k_left - (2 * q + h) * BK);
  }
#pragma unroll 1
  for (int q = 0; q < 2; q++) {
    k_tail_requests<MI>(sa + q * A_PAIR, a_tail + q * 128, a_off, a_k, 2 * BK, k_left - q * 2 * BK);
#pragma unroll
    for (int h = 0; h < (TB ? 1 : 2); h++)
      k_tail_requests<NB>(sb + q * B_PAIR + h * (B_PAIR / 2), b_tail + (TB ? q * 128 : (2 * q + h) * b_step), b_off, b_k,
                          TB ? 2 * BK : BK, k_left - (2 * q + h) * BK);
  }
}

// GATED: silu(A . B^T) * (A . up^T) of two weights [N,K]: the left half of a tile's columns are columns of B, the right half
// the same columns of `up`, so each wave column has one of the two products (bf16, one pass, a single GEMM).
template <int ES, bool TB, int MI, int NJ, bool GATED = false> __device__ __forceinline__ void w4_body(GemmParams p, const void *up = nullptr) {
  static_assert(!GATED || (TB && ES == 2), "gated: bf16 weights stored [N,K]");
  // B stored [N,K]: bf16 only.  (The same loop for 8-bit operands -- plain 16-byte fragment reads in place of the
  // transposing ones -- was measured against [K,N] on one board and is no faster: 166.9-168.9 against 167.2-168.6 us
  // for the 4096 x 4096 x 11008 layer; an 8-bit weight stored [N,K] is copied once instead.)
  static_assert(!TB || ES == 2, "B stored [N,K]: bf16 only");
  typedef W4Ring<ES, TB, MI, NJ> Ring;
  constexpr int BM = 32 * MI, BN = 32 * NJ, BK = 64 / ES, NB = TB ? NJ : NJ / 2;
  constexpr int A_PAIR = BM * 128, B_PAIR = BN * 128, RING = Ring::DA * A_PAIR + Ring::DB * B_PAIR;
  constexpr int DUMP_WAVE = 16 * MI * W4_DUMP_PITCH, EPILOGUE = 4 * DUMP_WAVE + 3 * 256 * 4;
  constexpr int CN = GATED ? BN / 2 : BN; // columns of C
  constexpr int B_ROW = BN * ES, B_CPR = B_ROW / 16, RG = ES == 2 ? 4 : 8; // B stored [K,N]: bytes and chunks of a k-row, k-rows per transposing read
#ifdef GCMI_W4_TIMING
  const long long wall_entry = wall_clock64();
  float *const timing_out = p.partial;
#endif
  // one array: the rings, afterwards the waves' accumulator regions and the column parameters behind them
  __shared__ __align__(1024) char smem[RING > EPILOGUE ? RING : EPILOGUE];
  float *colp = reinterpret_cast<float *>(smem + 4 * DUMP_WAVE);

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int r16 = lane & 15, g16 = lane >> 4;

  const int tiles_m = (int)((p.M + BM - 1) / BM), tiles_n = (int)((p.N + CN - 1) / CN); // edge tiles stick out
  int tm, tn;
  tile_of_block(blockIdx.x, gridDim.x, tiles_m, tiles_n, p.group_m, tm, tn);
  // integer division runs on the vector unit; the operand addresses below must be in scalar registers
  tm = __builtin_amdgcn_readfirstlane(tm), tn = __builtin_amdgcn_readfirstlane(tn);
  const int64_t m0 = (int64_t)tm * BM, n0 = (int64_t)tn * CN;
  const int64_t lda_b = p.lda * ES, ldb_b = p.ldb * ES;
  const int64_t b_step = TB ? 64 : BK * ldb_b; // from k-block to k-block
  // (a row of A is shorter than 2^31 bytes, so K fits 32 bits)
  const int all_groups = (int)((p.K + 4 * BK - 1) / (4 * BK));
  int k_left = (int)(p.K & (4 * BK - 1)), groups = all_groups;
  int64_t k_first = 0; // first k of this workgroup
  if (p.splits > 1) {
    // K slices: blockIdx.y is the slice, whole groups each (they differ by at most one); its f32 sums go
    // to the workspace as they are, the second kernel adds the slices and runs the epilogue
    const int slice = blockIdx.y;
    const int g0 = (int)((int64_t)slice * all_groups / p.splits), g1 = (int)((int64_t)(slice + 1) * all_groups / p.splits);
    k_first = (int64_t)g0 * 4 * BK, groups = g1 - g0;
    k_left = g1 == all_groups ? k_left : 0;
    p.C = p.partial + (int64_t)slice * p.M * p.N, p.ldc = p.N, p.out_dt = DT_F32;
    p.bias = nullptr, p.act = ACT_NONE, p.residual = nullptr;
  } else {
    const int64_t bz = blockIdx.y; // strided batch
    p.A = reinterpret_cast<const char *>(p.A) + bz * p.a_bs * ES;
    p.B = reinterpret_cast<const char *>(p.B) + bz * p.b_bs * ES;
    p.C = reinterpret_cast<char *>(p.C) + bz * p.c_bs * (p.out_dt == DT_BF16 ? 2 : 4);
    if (p.residual)
      p.residual = reinterpret_cast<const char *>(p.residual) + bz * p.c_bs * (p.residual_dt == DT_BF16 ? 2 : 4);
  }

  // Per-lane source offsets of the wave's DMA instructions, 1 KiB each: 8 rows by 128 bytes of A (or of B stored [N,K]), the
  // chunk that fills position c of row r is c ^ (r / 2 % 8); k-rows of a block of B stored [K,N].  An edge tile's rows past
  // M and columns past N are fetched from the last row / the last 16-byte chunk inside (N is a multiple of the
  // chunk's columns): their products land in accumulators that the epilogue never stores.
  const int rows_in = (int)min((int64_t)BM, p.M - m0), cols_in = (int)min((int64_t)CN, p.N - n0);
  // k-row k of B keeps chunk c at c ^ b_swz(k): the RG k-rows that a transposing read takes lie in different banks
  // (192 columns: rows of 384 bytes, k and k + 1 lie half the banks apart by themselves)
  auto b_swz = [](int k) { return BN == 192 ? ((k >> 1) & 1) * 4 : ES == 2 ? (k % 4) * 4 : BN == 256 ? (k % 8) * 2 : ((k % 8) >> 1) * 2; };
  int a_off[8] = {}, b_off[8] = {}, a_k[MI], b_k[NB]; // *_k: the first k of the lane's 16 bytes inside a pair / block
#pragma unroll
  for (int i = 0; i < MI; i++) {
    const int row = (wave * MI + i) * 8 + lane / 8, c = (lane % 8) ^ ((row >> 1) & 7);
    a_off[i] = (int)(min(row, rows_in - 1) * lda_b + c * 16);
    a_k[i] = c * 16 / ES;
  }
#pragma unroll
  for (int i = 0; i < NB; i++) {
    if constexpr (TB) {
      const int row = (wave * NB + i) * 8 + lane / 8, c = (lane % 8) ^ ((row >> 1) & 7);
      b_off[i] = (int)(min(GATED ? row % CN : row, cols_in - 1) * ldb_b + c * 16);
      b_k[i] = c * 16 / ES;
    } else {
      const int at = (wave * NB + i) * 64 + lane, krow = at / B_CPR;
      b_off[i] = (int)(krow * ldb_b + min((at % B_CPR) ^ b_swz(krow), cols_in * ES / 16 - 1) * 16);
      b_k[i] = krow;
    }
  }
  typedef int i32x8_t __attribute__((ext_vector_type(8)));
  i32x8_t a_src, b_src;
#pragma unroll
  for (int i = 0; i < 8; i++)
    a_src[i] = a_off[i], b_src[i] = b_off[i];
  // fragment addresses: A tile `it` = rows wm*16*MI + 16*it .., B tile `jt` = columns wn*16*NJ + 16*jt ..
  const uint32_t lds0 = (uint32_t)(uintptr_t)(GCMI_LDS char *)smem, lds_b = lds0 + Ring::DA * A_PAIR;
  i32x2_t a_ld;
  i32x4_t b_ld = {0, 0, 0, 0};
  {
    const int row_a = wm * 16 * MI + r16, row_b = wn * 16 * NJ + r16;
#pragma unroll
    for (int h = 0; h < 2; h++) {
      a_ld[h] = (int)(lds0 + row_a * 128 + (((4 * h + g16) ^ ((row_a >> 1) & 7)) << 4));
      if (TB)
        b_ld[h] = (int)(lds_b + row_b * 128 + (((4 * h + g16) ^ ((row_b >> 1) & 7)) << 4));
    }
    if (!TB) {
      // the 16 lanes of a group hand the transposing read RG k-rows x 16 columns in 8-byte pieces (bf16: k row
      // lane%16/4, 4 columns at lane%4; int8: k row lane%16/2, 8 columns at lane%2) and get back column lane%16;
      // tiles 2j and 2j + 1 differ in a chunk bit that b_swz leaves alone
      const int kk = ES == 2 ? (r16 >> 2) : (r16 >> 1), cc = ES == 2 ? (r16 & 3) : (r16 & 1);
#pragma unroll
      for (int j = 0; j < NJ / 2; j++) {
        const int chunk = ES == 2 ? (wn * NJ + 2 * j) * 2 + (cc >> 1) : wn * NJ + 2 * j;
        const int sub = ES == 2 ? (cc & 1) * 8 : cc * 8;
        b_ld[j] = (int)(lds_b + (2 * RG * g16 + kk) * B_ROW + ((chunk ^ b_swz(kk)) << 4) + sub);
      }
    }
  }

  // column parameters of this tile: 256 threads, one column each
  float cp_bias = -0.0f, cp_scale = 1.0f; // an absent bias adds nothing, not even to -0.0
  int cp_cs = 0;
  if (tid < cols_in) {
    if (p.bias)
      cp_bias = p.bias_dt == DT_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p.bias)[n0 + tid])
                                     : reinterpret_cast<const float *>(p.bias)[n0 + tid];
    if (ES == 1) {
      if (p.scale)
        cp_scale = p.scale[n0 + tid];
      if (p.colsum)
        cp_cs = p.comp * p.colsum[n0 + tid];
    }
  }

  // (inputs of the assembly in scalar registers)
  const char *const a0 = reinterpret_cast<const char *>(p.A) + m0 * lda_b + k_first * ES;
  // (gated: waves 0 and 1 request the rows of the left half, 2 and 3 those of the right one)
  const char *const b0 = reinterpret_cast<const char *>(GATED && wave >= 2 ? up : p.B) + (TB ? n0 * ldb_b + k_first * ES : n0 * ES + k_first * ldb_b);
  uint64_t a_ptr = (uint64_t)a0, b_ptr = (uint64_t)b0;
  int pairs = __builtin_amdgcn_readfirstlane(2 * groups);
  const int tail_group = __builtin_amdgcn_readfirstlane(k_left);
  const uint32_t a_dma = lds0 + (uint32_t)(wave * MI * 1024), b_dma = lds_b + (uint32_t)(wave * NB * 1024);
  const uint32_t a_xor = p.a_xor;
  // where this lane writes its accumulators for the epilogue: row lane%16 (+ 16*it), 16-byte chunk lane/16 (+ 4*jt)
  // of the wave's region
  const uint32_t dump_ld = lds0 + (uint32_t)wave * DUMP_WAVE + (uint32_t)(r16 * W4_DUMP_PITCH + g16 * 16);

#define GCMI_W4_FILL(TEXT)                                                                                            \
  asm volatile(TEXT : "+{s[40:41]}"(a_ptr), "+{s[42:43]}"(b_ptr)                                                      \
               : "{v[0:7]}"(a_src), "{v[8:15]}"(b_src), "{s[44:45]}"(b_step), "{s46}"(pairs), "{s47}"(a_dma),         \
                 "{s51}"(b_dma), "{s50}"(tail_group)                                                                  \
               : "memory", "scc", "s49")
#define GCMI_W4_MAIN(TEXT, CLOBBERS)                                                                                  \
  asm volatile(TEXT : "+{s[40:41]}"(a_ptr), "+{s[42:43]}"(b_ptr), "+{s46}"(pairs)                                     \
               : "{v[0:7]}"(a_src), "{v[8:15]}"(b_src), "{v[16:17]}"(a_ld), "{v[20:23]}"(b_ld),                       \
                 "{s[44:45]}"(b_step), "{s47}"(a_dma), "{s51}"(b_dma), "{s48}"(a_xor), "{s50}"(tail_group), "{v28}"(dump_ld) \
               : "memory", "scc", "s49", "s52", "s53", "s54", "s55", "s56", CLOBBERS)
#define GCMI_W4_OF(STEP)                                                                                              \
  if constexpr (ES == 1 && NJ == 8) STEP(I8_8x8, 8x8)                                                                 \
  else if constexpr (ES == 1 && MI == 8) STEP(I8_8x4, 8x4)                                                            \
  else if constexpr (ES == 1 && MI == 6) STEP(I8_6x4, 6x4)                                                            \
  else if constexpr (ES == 1) STEP(I8_4x4, 4x4)                                                                       \
  else if constexpr (TB && NJ == 8) STEP(BF16_TB_8x8, 8x8)                                                            \
  else if constexpr (TB && NJ == 6) STEP(BF16_TB_8x6, 8x6)                                                            \
  else if constexpr (TB && MI == 8) STEP(BF16_TB_8x4, 8x4)                                                            \
  else if constexpr (TB && MI == 6) STEP(BF16_TB_6x4, 6x4)                                                            \
  else if constexpr (TB) STEP(BF16_TB_4x4, 4x4)                                                                       \
  else if constexpr (NJ == 8) STEP(BF16_8x8, 8x8)                                                                     \
  else if constexpr (NJ == 6) STEP(BF16_8x6, 8x6)                                                                     \
  else if constexpr (MI == 8) STEP(BF16_8x4, 8x4)                                                                     \
  else if constexpr (MI == 6) STEP(BF16_6x4, 6x4)                                                                     \
  else STEP(BF16_4x4, 4x4)
#define GCMI_W4_STEP_FILL(NAME, TILES) GCMI_W4_FILL(GCMI_W4_FILL_##NAME);
#define GCMI_W4_STEP_MAIN(NAME, TILES) GCMI_W4_MAIN(GCMI_W4_ASM_##NAME, GCMI_W4_CLOBBERS_##TILES);
  if (tail_group) {
    const int64_t k_full = p.K - k_left - k_first;
    w4_request_k_tail<ES, TB, MI, NJ>(smem, wave, lane, a0 + k_full * ES, b0 + (TB ? k_full * ES : k_full * ldb_b), b_step, k_left,
                                      a_off, b_off, a_k, b_k);
  }
  GCMI_W4_OF(GCMI_W4_STEP_FILL)
#ifdef GCMI_W4_TIMING // measurement builds: core clock cycles and 100 MHz ticks spent in the main loop
  const long long tick0 = clock64(), wall0 = wall_clock64();
#endif
  GCMI_W4_OF(GCMI_W4_STEP_MAIN)
#undef GCMI_W4_OF
#undef GCMI_W4_STEP_FILL
#undef GCMI_W4_STEP_MAIN
#undef GCMI_W4_FILL
#undef GCMI_W4_MAIN
#ifdef GCMI_W4_TIMING
  const long long tick1 = clock64(), wall1 = wall_clock64();
#endif
  if constexpr (GATED) {
    const char *const gate = smem + 2 * wm * DUMP_WAVE, *const other = gate + DUMP_WAVE;
    __syncthreads();
    w4_gated_half<16 * MI, 16 * NJ>(p, 0, m0, n0, wm, wn, lane, gate, other, rows_in, cols_in);
    if constexpr (NJ > 4) {
      __syncthreads(); // the other wave has read this one's region
      if constexpr (NJ == 8)
        asm volatile(GCMI_W4_ASM_DUMP_HI_8x8 : : "{v28}"(dump_ld) : "memory");
      else
        asm volatile(GCMI_W4_ASM_DUMP_HI_8x6 : : "{v28}"(dump_ld) : "memory");
      __syncthreads();
      w4_gated_half<16 * MI, 16 * NJ>(p, 1, m0, n0, wm, wn, lane, gate, other, rows_in, cols_in);
    }
    return;
  }
  // the column parameters were requested before the main loop and are first needed here
  colp[tid] = cp_bias;
  if (ES == 1) {
    colp[256 + tid] = cp_scale;
    reinterpret_cast<int *>(colp)[512 + tid] = cp_cs;
  }
  __syncthreads();

  const int out_kind = p.out_dt == DT_BF16 ? 0 : ((ES == 1 && p.out_dt == DT_S32) ? 2 : 1);
  const int kind = (out_kind == 2 ? (int)ACT_NONE : p.act) + 8 * out_kind;
  const char *dump = smem + wave * DUMP_WAVE;
  // a tile that sticks out of C takes the same code with every row and lane tested against the edge
  const bool edge_tile = rows_in < BM || cols_in < BN; // the same for the whole workgroup
  if (edge_tile)
    w4_epilogue_half_any<ES, true, 16 * MI, 16 * NJ>(p, kind, 0, m0, n0, wm, wn, lane, dump, colp, rows_in, cols_in);
  else
    w4_epilogue_half_any<ES, false, 16 * MI, 16 * NJ>(p, kind, 0, m0, n0, wm, wn, lane, dump, colp, BM, BN);
  if constexpr (NJ > 4) {
    // the right part: the accumulators of column tiles 4 and up are still where the main loop left them
    static_assert(MI == 8 && (NJ == 8 || NJ == 6), "the dumps there are");
    if constexpr (NJ == 8)
      asm volatile(GCMI_W4_ASM_DUMP_HI_8x8 : : "{v28}"(dump_ld) : "memory");
    else
      asm volatile(GCMI_W4_ASM_DUMP_HI_8x6 : : "{v28}"(dump_ld) : "memory");
    if (edge_tile)
      w4_epilogue_half_any<ES, true, 16 * MI, 16 * NJ>(p, kind, 1, m0, n0, wm, wn, lane, dump, colp, rows_in, cols_in);
    else
      w4_epilogue_half_any<ES, false, 16 * MI, 16 * NJ>(p, kind, 1, m0, n0, wm, wn, lane, dump, colp, BM, BN);
  }
#ifdef GCMI_W4_TIMING
  const long long wall_issued = wall_clock64();
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (timing_out && tid == 0 && blockIdx.x < 256) {
    long long *t = reinterpret_cast<long long *>(timing_out) + 8 * blockIdx.x;
    t[0] = tick1 - tick0, t[1] = wall1 - wall0, t[2] = wall0 - wall_entry, t[3] = wall_issued - wall1, t[4] = wall_clock64() - wall_issued;
    t[5] = wall_entry;
  }
#endif
}

template <int ES, bool TB = false> __global__ __launch_bounds__(256, 1) void gemm_tile256_w4_kernel(GemmParams p) { w4_body<ES, TB, 8, 8>(p); }
// 128, 192 or 256 rows by 128 columns, 256 rows by 192
template <bool TB, int ES, int MI, int NJ = 4> __global__ __launch_bounds__(256, 1) void gemm_tall_kernel(GemmParams p) { w4_body<ES, TB, MI, NJ>(p); }

template <bool TB, int ES> static int launch_tall(const GemmParams &p, int rows, int cols, dim3 grid, hipStream_t stream) {
  if (rows == 128 && cols == 128)
    hipLaunchKernelGGL((gemm_tall_kernel<TB, ES, 4>), grid, dim3(256), 0, stream, p);
  else if (rows == 192 && cols == 128)
    hipLaunchKernelGGL((gemm_tall_kernel<TB, ES, 6>), grid, dim3(256), 0, stream, p);
  else if (rows == 256 && cols == 128)
    hipLaunchKernelGGL((gemm_tall_kernel<TB, ES, 8>), grid, dim3(256), 0, stream, p);
  else if constexpr (ES == 2)
    hipLaunchKernelGGL((gemm_tall_kernel<TB, ES, 8, 6>), grid, dim3(256), 0, stream, p);
  else
    return 2;
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

// Four results of row m, columns n .. n+3, from their f32 sums: the rounding points of a bf16 graph (after the
// matmul and after every op, lib/gc/Transforms/Pipeline.cpp:79-95), or one f32 epilogue.
__device__ __forceinline__ f32x4_t epilogue_bias4(const GemmParams &p, int64_t n) {
  f32x4_t b = {0.f, 0.f, 0.f, 0.f};
  if (p.bias)
#pragma unroll
    for (int c = 0; c < 4; c++)
      b[c] = p.bias_dt == DT_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p.bias)[n + c])
                                  : reinterpret_cast<const float *>(p.bias)[n + c];
  return b;
}
__device__ __forceinline__ void epilogue_store4(const GemmParams &p, const f32x4_t &v, int64_t m, int64_t n, const f32x4_t &b4) {
  float o32[4];
  uint16_t o16[4];
#pragma unroll
  for (int c = 0; c < 4; c++) {
    const float b = b4[c];
    float x = v[c], r = 0.0f;
    if (p.residual)
      r = p.residual_dt == DT_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p.residual)[m * p.ldr + n + c])
                                   : reinterpret_cast<const float *>(p.residual)[m * p.ldr + n + c];
    if (p.out_dt == DT_BF16) {
      x = round_bf16(x);
      if (p.bias)
        x = round_bf16(x + b);
      if (p.act != ACT_NONE)
        x = round_bf16(apply_act_of_bf16(x, p.act));
      if (p.residual)
        x = round_bf16(x + r);
    } else {
      if (p.bias)
        x = x + b;
      x = apply_act(x, p.act);
      if (p.residual) { // kept apart from the activation's last multiply: the sum equals a separate add
#pragma clang fp contract(off)
        x = x + r;
      }
    }
    o32[c] = x;
    o16[c] = f32_to_bf16_bits(x);
  }
  if (p.out_dt == DT_BF16)
    *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(p.C) + m * p.ldc + n) =
        make_uint2(o16[0] | ((uint32_t)o16[1] << 16), o16[2] | ((uint32_t)o16[3] << 16));
  else
    *reinterpret_cast<f32x4_t *>(reinterpret_cast<float *>(p.C) + m * p.ldc + n) = f32x4_t{o32[0], o32[1], o32[2], o32[3]};
}

// Second pass of split-K: out = epilogue(sum over slices of the f32 partials), slices added in ascending
// order (deterministic), the same rounding points as the fused epilogue.  One thread per 4 columns; the
// loads of eight slices are in flight together.
template <int ACT> __global__ __launch_bounds__(256) void gemm_splitk_reduce_kernel(GemmParams p) {
  const int64_t n4 = p.N / 4, idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (idx >= p.M * n4)
    return;
  const int64_t m = idx / n4, n = (idx % n4) * 4, sl = p.M * p.N;
  const float *src = p.partial + m * p.N + n;
  f32x4_t a = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < p.splits; s0 += 8) {
    f32x4_t b[8];
#pragma unroll
    for (int u = 0; u < 8; u++)
      b[u] = s0 + u < p.splits ? *reinterpret_cast<const f32x4_t *>(src + (s0 + u) * sl) : f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (s0 + u < p.splits) {
        if (s0 + u == 0)
          a = b[u];
        else
          a[0] += b[u][0], a[1] += b[u][1], a[2] += b[u][2], a[3] += b[u][3];
      }
  }
  float bias4[4] = {0.f, 0.f, 0.f, 0.f};
  if (p.bias) {
#pragma unroll
    for (int e = 0; e < 4; e++)
      bias4[e] = p.bias_dt == DT_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p.bias)[n + e])
                                      : reinterpret_cast<const float *>(p.bias)[n + e];
  }
  uint16_t o16[4];
  float o32[4];
#pragma unroll
  for (int e = 0; e < 4; e++) {
    float x = a[e], r = 0.0f;
    if (p.residual)
      r = p.residual_dt == DT_BF16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t *>(p.residual)[m * p.ldr + n + e])
                                   : reinterpret_cast<const float *>(p.residual)[m * p.ldr + n + e];
    if (p.out_dt == DT_BF16) { // bf16 graph: round after the matmul and after every bf16 op
      x = round_bf16(x);
      if (p.bias)
        x = round_bf16(x + bias4[e]);
      if (ACT != ACT_NONE)
        x = round_bf16(apply_act_of_bf16(x, ACT));
      if (p.residual)
        x = round_bf16(x + r);
    } else {
      if (p.bias)
        x = x + bias4[e];
      x = act_const<ACT>(x);
      if (p.residual) { // kept apart from the activation's last multiply: the sum equals a separate add
#pragma clang fp contract(off)
        x = x + r;
      }
    }
    o32[e] = x;
    o16[e] = f32_to_bf16_bits(x);
  }
  if (p.out_dt == DT_BF16)
    *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(p.C) + m * p.ldc + n) =
        make_uint2(o16[0] | ((uint32_t)o16[1] << 16), o16[2] | ((uint32_t)o16[3] << 16));
  else
    *reinterpret_cast<f32x4_t *>(reinterpret_cast<float *>(p.C) + m * p.ldc + n) = f32x4_t{o32[0], o32[1], o32[2], o32[3]};
}

// second pass of every K-sliced GEMM: one thread per four outputs, the activation as a template argument
static void launch_splitk_reduce(const GemmParams &p, hipStream_t stream) {
  if (p.leave_splits > 1 && p.leave_splits == p.splits) {
    *p.left = 1;
    return;
  }
  const dim3 grid((unsigned)((p.M * (p.N / 4) + 255) / 256)), block(256);
  switch (p.act) {
  case ACT_RELU:
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel<ACT_RELU>, grid, block, 0, stream, p);
    break;
  case ACT_GELU_ERF:
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel<ACT_GELU_ERF>, grid, block, 0, stream, p);
    break;
  case ACT_GELU_TANH:
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel<ACT_GELU_TANH>, grid, block, 0, stream, p);
    break;
  case ACT_SIGMOID:
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel<ACT_SIGMOID>, grid, block, 0, stream, p);
    break;
  default:
    hipLaunchKernelGGL(gemm_splitk_reduce_kernel<ACT_NONE>, grid, block, 0, stream, p);
    break;
  }
}

// 128 columns, 128 rows or more: gemm_tile128.hpp
static constexpr int T128_B = 128, T128_KB = 64, T128_NST = 4;

// Whether tiles of rows x cols run on the kernel that puts two of them on a compute unit, or alone on the 4-wave kernels' hand-placed loop.
// Two 128 x 128 tiles per compute unit only where there are more than a round of them, or two groups of K or less, which are
// set-up and epilogue mostly.  Else the hand-placed loop with its deeper ring, the whole LDS to itself, us, two per unit / this,
// weights from memory: 1000 x 4096, K 4096 [N,K] 48.2 / 37.2, 2048^3 27.8 / 23.7, 1422 x 2384, K 1280 [N,K] 16.3 / 12.9, 1086 x 144,
// K 272 7.6 / 7.4, 8-bit 1024 x 4096, K 4096 31.5 / 26.9; but 746 x 944, K 160 7.4 / 7.6, 8-bit 1425 x 1168, K 208 7.9 / 8.3, and in more
// than a round 2498 x 2544, K 512 13.3 / 14.2.
static inline bool tile128_in_pairs(int es, int rows, int cols, int64_t K, int splits, int64_t workgroups) {
  return rows == 128 && cols == 128 && (workgroups > gcmi_num_cus() || K * es <= 512 * (int64_t)(splits > 1 ? splits : 1));
}

// How many k-blocks (64 bytes of K per row) of both operands the LDS rings of the 4-wave kernel of rows x cols hold.
template <int ES, bool TB, int MI, int NJ> constexpr int w4_ring_blocks() {
  return 2 * (W4Ring<ES, TB, MI, NJ>::DA < W4Ring<ES, TB, MI, NJ>::DB ? W4Ring<ES, TB, MI, NJ>::DA : W4Ring<ES, TB, MI, NJ>::DB);
}
template <int ES, bool TB> static inline int w4_ring_blocks(int rows, int cols) {
  if (cols == 128)
    return rows == 128 ? w4_ring_blocks<ES, TB, 4, 4>() : rows == 192 ? w4_ring_blocks<ES, TB, 6, 4>() : w4_ring_blocks<ES, TB, 8, 4>();
  if constexpr (ES == 2)
    if (cols == 192)
      return w4_ring_blocks<ES, TB, 8, 6>();
  return w4_ring_blocks<ES, TB, 8, 8>();
}
// ... of the kernel that runs tiles of 128 x 128 to 256 x 192
template <int ES> static inline int tile128_stages(int rows, int cols, int64_t K, int trans_b, int splits, int64_t workgroups) {
  if (tile128_in_pairs(ES, rows, cols, K, splits, workgroups))
    return T128_NST;
  if constexpr (ES == 2)
    if (trans_b)
      return w4_ring_blocks<2, true>(rows, cols);
  return w4_ring_blocks<ES, false>(rows, cols);
}

} // namespace gcmi
extern "C" int gcmi_launch_tile128(const gcmi::GemmParams *p, int es, int rows, int cols, unsigned grid_x, unsigned grid_y, hipStream_t stream);
namespace gcmi {

// Host-side launch of the 256x256 tile kernels for one element size.
// want != null: nothing is launched; *want receives the floats of workspace this call would use if it had them, *optional whether
// it is one that the taller tiles brought to slices: without them it runs in one pass, so no entry point may refuse it for
// want of a workspace.
// cfg != null: receives what was (or would be) chosen.
// Estimates behind the choice of tile and K slices for bf16 problems that do not fill the GPU with 256 x 256 tiles,
// in microseconds, fitted to graph-replayed timings on a 256-CU board (load = workgroups / compute units).  One ring
// group = 128 elements of K.  The rates grow with the load because the board lowers its clock as more of it works.
static inline double gcmi_us_per_group_256(double load) { // one workgroup per compute unit
  if (load <= 0.25)
    return 1.94;
  if (load <= 0.5)
    return 1.94 + 0.16 * (load - 0.25) / 0.25;
  if (load <= 1.0)
    return 2.1 + 0.65 * (load - 0.5) / 0.5;
  return 2.75;
}
// Taller tiles of 128 columns (one workgroup per compute unit): fewer fragment reads per product than 128 rows, so where 128
// rows make more than a round and 192 or 256 do not, they are ahead; where 128 rows fit one round they stay.  These rates, and those of
// 128 rows up to a load of 1, were fitted to a main loop that the compiler had scheduled.  The hand-placed one is about an
// eighth faster (GCMI_TILE_COSTS below rates it), which the comparison with K slices and with 256 x 256 tiles here does not have yet.
static inline double gcmi_us_per_group_tall(int rows) { return rows == 192 ? 1.5 : 1.85; }
static inline double gcmi_us_fixed_tall(int rows, int es) { return (rows == 192 ? 5.0 : 6.0) + (es == 1 ? 1.0 : 0.0); } // (8-bit: the longer epilogue, alone on its unit)
// A long K beside wide weights costs 128 rows more per group than the estimate has, which was fitted to weights that the
// last-level cache holds from call to call (256 MiB; 1.04 us at any K): from memory, as a model's weights come, a group takes
// 1.38.  Up to a K of 8192 the choice is the same either way; past it taller tiles, which read them fewer times, are ahead.
// 1000 x 4096 [N,K], one pass of 128 rows / two slices of 256, from memory (from the cache), us: K 6144 71.2 / 72.3 (57 / 68), 8192
// 82.7 / 85.2 (68 / 83), 9728 107 / 102 (87 / 96), 11008 128 / 112 (105 / 106), 12288 139 / 122 (110 / 116), 14336 159 / 140, 16384 175 /
// 159, 22016 249 / 214; [K,N] the two meet at 11008 (122 / 124) and 22016 has 234 / 219.  Random sizes of more than 256 rows and 512
// columns or more, against the rules without this and without taller tiles: K 8200 to 24576 90 of them 1.13 times from the cache,
// 1.15 from memory (0.87 to 1.6), K to 60000 24 of them 1.17 and 1.16.  Fewer rows or columns have weights or results so small that
// it only made more slices of them: 26 sizes 0.95, down to 0.7.
static inline double gcmi_us_per_group_128_long_k(int64_t K) {
  return K <= 8192 ? 0.0 : K >= 11008 ? 0.27 : 0.27 * (double)(K - 8192) / 2816.0;
}
static inline double gcmi_us_per_group_128(double load) { // up to two workgroups per compute unit
  if (load <= 0.25)
    return 0.85;
  if (load <= 1.0)
    return 0.85 + 0.27 * (load - 0.25) / 0.75;
  if (load <= 2.0) // as soon as some compute units hold two workgroups, those set the pace
    return 1.9 + 0.27 * (load - 1.0);
  return 2.17;
}
static constexpr double GCMI_US_FIXED_256 = 8.0, GCMI_US_FIXED_128 = 3.7; // launch, ring fill, epilogue
static constexpr double GCMI_US_SECOND_PASS = 3.0;     // the second kernel of a K-sliced product
static constexpr double GCMI_US_PER_SLICE_MOUT = 1.7;  // partial sums written and read back, per slice and 2^20 outputs
static constexpr double GCMI_ONE_PASS_MARGIN = 0.9;    // slices must win by this factor
// bf16 problems that would take 256 x 256 tiles in one pass: the time of one pass by tile, us, fitted to 184 random graph-replayed ones
// with the weights from memory (500 to 4500 rows, 1500 to 11008 columns, K 64 to 6000, up to 2.7 rounds of large tiles; rms
// error 9 to 12 %).  A launch, per round of workgroups (one per compute unit; two of 128 x 128) a start and an epilogue, per group of
// 128 k its rounds and, as the clock and the memory system notice, its tiles per compute unit, and 2^20 results stored.
struct GemmTileCost {
  int rows, cols, per_cu;
  double launch, round, group_round, group_load, mout;
};
static constexpr GemmTileCost GCMI_TILE_COSTS[] = {
    {256, 256, 1, 2.2, 9.3, 1.46, 1.29, 0.05}, {256, 192, 1, 2.9, 7.3, 1.45, 0.65, 0.19}, {256, 128, 1, 3.1, 4.7, 0.93, 0.68, 0.09},
    {192, 128, 1, 3.7, 2.7, 1.01, 0.29, 0.31}, {128, 128, 2, 2.2, 2.2, 0.59, 0.93, 0.12}};
static inline double gcmi_us_tile(const GemmTileCost &t, int64_t M, int64_t N, int64_t batches, int groups, int n_cu) {
  const double load = (double)(((M + t.rows - 1) / t.rows) * ((N + t.cols - 1) / t.cols) * batches) / n_cu;
  const double rounds = ceil(load / t.per_cu);
  return t.launch + t.round * rounds + groups * (t.group_round * rounds + t.group_load * load) +
         t.mout * (double)M * (double)N * (double)batches / 1048576.0;
}
enum GemmPlan { PLAN_TILE256 = 0, PLAN_TILE128, PLAN_SLICES_SHORT_A, PLAN_SLICES_TILE256, PLAN_SLICES_TILE128 };
template <int ES>
static int launch_tile256(const GemmParams *pp, hipStream_t stream, int64_t *want = nullptr, GemmTileConfig *cfg = nullptr,
                          bool *optional = nullptr) {
  GemmParams p = *pp;
  if (want)
    *want = 0, *optional = false;
  const bool dry = want != nullptr || (cfg != nullptr && stream == (hipStream_t)-1);
  const int64_t ws_cap = want ? INT64_MAX : (p.partial ? p.partial_cap : 0);
  float *const ws = p.partial;
  const int tiles_m = (int)((p.M + G_BM - 1) / G_BM), tiles_n = (int)((p.N + G_BN - 1) / G_BN);
  const int64_t nblk = (int64_t)tiles_m * tiles_n;
  if (nblk <= 0 || nblk > 0x7fffffff)
    return 2;
  const int out_es = p.out_dt == DT_BF16 ? 2 : 4;
  auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  const int BK = G_KBYTES / ES;
  // fast path: whole tiles, 16-byte aligned rows, and a tile's rows reachable with 32-bit byte offsets
  const int KGROUP = 256 / ES; // K elements of one trip round the LDS ring
  const int res_es = p.residual_dt == DT_BF16 ? 2 : 4;
  // the kernels for whole tiles read four residual elements with one load
  const bool res_vec = !p.residual || (al16(p.residual) && (p.ldr * res_es) % 16 == 0);
  // K: whole 16-byte chunks; the 4-wave kernel and the 128 x 128 one take an incomplete last ring group themselves,
  // the others need whole groups
  const bool k_whole = p.K % KGROUP == 0;
  const bool aligned = p.K % (16 / ES) == 0 && p.K > 0 && al16(p.A) && al16(p.B) && al16(p.C) && res_vec &&
                       (p.lda * ES) % 16 == 0 && (p.ldb * ES) % 16 == 0 && (p.ldc * out_es) % 16 == 0 &&
                       p.lda * ES * G_BM < (int64_t)1 << 31 && p.ldb * ES * (p.trans_b ? G_BN : BK) < (int64_t)1 << 31;
  const bool fast_but_m = aligned && k_whole && p.N % G_BN == 0;
  if (p.trans_b && ES != 2)
    return 3;
  if (p.residual && (ES != 2 || (p.residual_dt != DT_BF16 && p.residual_dt != DT_F32) || p.out_dt == DT_S32))
    return 3;
  bool fast = fast_but_m && p.M % G_BM == 0;
  p.splits = 0;
  p.partial = nullptr;
  const int64_t nbatch = p.batch > 1 ? p.batch : 1;
  if (nbatch > 65535)
    return 2;
  if (nbatch == 1)
    p.a_bs = p.b_bs = p.c_bs = 0;
  else if (!((p.a_bs * ES) % 16 == 0 && (p.b_bs * ES) % 16 == 0 && (p.c_bs * out_es) % 16 == 0 &&
             (!p.residual || (p.c_bs * res_es) % 16 == 0)))
    fast = false; // every batch's operands must keep the alignment the fast path loads with
  // Any M, N and K whole numbers of 16-byte chunks: the 4-wave kernel still takes it; its edge tiles clamp their loads
  // and store what lies inside C.
  // A K of 64 bf16 or less under fewer than 32 rows stays with the bounds-checked kernel, which is no line by speed: 11.1 us there, 9.3
  // here (16 x 20000, K 64), since the 4-wave epilogue passes over rows outside C (before that 12.4; from K 65 on this one was ahead).
  const bool tiny = ES == 2 && !k_whole && p.K <= 64 && p.M < 32 && p.cfg_tile == 0;
  const bool ragged = !fast && !tiny && aligned && p.N % (16 / ES) == 0 && (p.M % G_BM != 0 || p.N % G_BN != 0 || !k_whole) &&
                      (nbatch == 1 || ((p.a_bs * ES) % 16 == 0 && (p.b_bs * ES) % 16 == 0 && (p.c_bs * out_es) % 16 == 0 &&
                                       (!p.residual || (p.c_bs * res_es) % 16 == 0)));
  if (p.group_m <= 0)
    p.group_m = 4;
  GemmTileConfig c{};
  c.bm = G_BM, c.bn = G_BN, c.split_k = 1, c.group_m = p.group_m, c.workgroups = (int32_t)nblk;
  c.from_attrs = (p.cfg_waves || p.cfg_split_k || p.cfg_tile == 256) ? 1 : 0;

  // What runs.  bf16 problems that fill the GPU with 256 x 256 tiles take those; smaller ones are given to more
  // workgroups, either by 128 x 128 tiles (two workgroups per compute unit: four times the workgroups), or by cutting
  // K into slices (one workgroup per tile and slice; f32 partial sums through the workspace and a small second
  // kernel; the slice count plays the part of the reference's KThreads, lib/gc/Analysis/MatmulConfigAnalysis.cpp:149-166),
  // or both; the estimates above decide.  A short A (M <= 128: decode-style shapes such as 32 x 4096 x 4096, whose
  // weights have to stream from HBM through all compute units) keeps the kernel that skips the empty 32-row blocks
  // of its tile and takes slices of unequal length, unless the 128 x 128 tiles are estimated faster (from 32 rows
  // on they are).  The 128 x 128 kernel cuts K itself (blockIdx.y = slice, whole ring groups, lengths differing by at
  // most one); the 256 x 256 kernel runs equal slices as a strided batch: batch = K slice, results f32 with
  // c_bs = M * N.  A caller's MatmulConfig replaces the choice.
  const bool batch_ok = nbatch == 1 || ((p.a_bs * ES) % 16 == 0 && (p.b_bs * ES) % 16 == 0 && (p.c_bs * out_es) % 16 == 0 &&
                                        (!p.residual || (p.c_bs * res_es) % 16 == 0));
  const bool t128_can = aligned && p.N % (16 / ES) == 0 && (ES == 2 ? p.out_dt != DT_S32 : !p.trans_b) && batch_ok;
  const bool slices_can = ES == 2 && fast_but_m && p.out_dt != DT_S32 && nbatch == 1; // the 256-wide kernels: whole column tiles
  const int n_cu = gcmi_num_cus();
  const int groups = (int)((p.K + KGROUP - 1) / KGROUP);
  struct Choice {
    int plan, splits, rows128; // rows of the 128-column tile
  };
  // The choice by the estimates, with slices whose partial sums fit `cap` floats.  taller: the tiles of 192 and 256 rows, and what
  // a long K costs those of 128, take part.
  auto choose = [&](bool taller, int64_t cap) -> Choice {
    Choice ch{PLAN_TILE256, 1, 128};
    const int64_t nblk128 = ((p.M + 127) / 128) * ((p.N + 127) / 128);
    const double mn = (double)p.M * (double)p.N / 1048576.0;
    const double w256 = (double)(nblk * nbatch) / n_cu, w128 = (double)(nblk128 * nbatch) / n_cu;
    double best = GCMI_US_FIXED_256 + gcmi_us_per_group_256(w256) * groups; // one pass, less than one round
    const bool small_tile = p.M >= 32 && t128_can; // shorter: most of a 128-row tile would be padding
    const double long_k = ES == 2 && taller && p.M > 256 && p.N >= 512 ? gcmi_us_per_group_128_long_k(p.K) : 0.0; // (of two workgroups on a compute unit, both)
    // taller tiles: at least two rows of them, in one round
    auto tall_tiles = [&](int rows) { return ((p.M + rows - 1) / rows) * ((p.N + 127) / 128) * nbatch; };
    auto fits = [&](int s) { return (int64_t)s * p.M * p.N <= cap; };
    if (small_tile) {
      const double t = GCMI_US_FIXED_128 + (gcmi_us_per_group_128(w128) + (w128 <= 1.0 ? 1 : 2) * long_k) * groups * (double)((nblk128 * nbatch + 2 * n_cu - 1) / (2 * n_cu));
      if (t < best)
        best = t, ch.plan = PLAN_TILE128;
      for (int rows = 192; taller && rows <= 256; rows += 64) {
        const double u = gcmi_us_fixed_tall(rows, ES) + gcmi_us_per_group_tall(rows) * groups;
        if (p.M > rows && tall_tiles(rows) <= n_cu && u < best)
          best = u, ch = {PLAN_TILE128, 1, rows};
      }
    }
    best *= GCMI_ONE_PASS_MARGIN;
    if (ES == 2 && nbatch == 1 && (small_tile || p.M > 128)) {
      for (int s = 2; s <= groups && fits(s); s++) {
        const double through_memory = GCMI_US_SECOND_PASS + GCMI_US_PER_SLICE_MOUT * s * mn;
        if (slices_can && p.M > 128 && groups % s == 0 && nblk * s <= n_cu) {
          const double t = GCMI_US_FIXED_256 + gcmi_us_per_group_256(w256 * s) * (groups / s) + through_memory;
          if (t < best)
            best = t, ch = {PLAN_SLICES_TILE256, s, 128};
        }
        if (small_tile && nblk128 * s <= 2 * n_cu) {
          const double t = GCMI_US_FIXED_128 + (gcmi_us_per_group_128(w128 * s) + (nblk128 * s <= n_cu ? 1 : 2) * long_k) * ((groups + s - 1) / s) + through_memory;
          if (t < best)
            best = t, ch = {PLAN_SLICES_TILE128, s, 128};
        }
      }
      double tall_best = best * (ch.splits > 1 ? GCMI_ONE_PASS_MARGIN : 1.0); // against other slices they too must be clearly ahead
      for (int s = 2; taller && small_tile && s <= groups && fits(s); s++)
        for (int rows = 192; rows <= 256; rows += 64) {
          const double t = gcmi_us_fixed_tall(rows, ES) + gcmi_us_per_group_tall(rows) * ((groups + s - 1) / s) + GCMI_US_SECOND_PASS +
                           GCMI_US_PER_SLICE_MOUT * s * mn;
          if (p.M > rows && tall_tiles(rows) * s <= n_cu && t < tall_best)
            tall_best = best = t, ch = {PLAN_SLICES_TILE128, s, rows};
        }
    }
    if (nbatch == 1 && p.M <= 128 && slices_can && nblk * 2 <= n_cu) { // a short A: 1.35 (32 rows) to 2 us (128) per group
      const double per_group = 1.35 + 0.65 * (double)((p.M + 31) / 32 - 1) / 3.0;
      const int smax = n_cu / (int)nblk < groups ? n_cu / (int)nblk : groups;
      for (int s = 2; s <= smax && fits(s); s++) {
        const double t = 7.0 + per_group * ((groups + s - 1) / s) + GCMI_US_PER_SLICE_MOUT * s * mn;
        if (t < best)
          best = t, ch = {PLAN_SLICES_SHORT_A, s, 128};
      }
    }
    return ch;
  };
  Choice chosen{PLAN_TILE256, 1, 128};
  if (p.cfg_tile == 128) {
    if (t128_can && ((p.M + 127) / 128) * ((p.N + 127) / 128) <= 0x7fffffff)
      chosen.plan = PLAN_TILE128, c.from_attrs = 1;
  } else if (p.cfg_tile == 256) {
    if (slices_can && p.cfg_split_k > 1) {
      chosen.splits = p.cfg_split_k < groups ? p.cfg_split_k : groups;
      chosen.plan = p.M > 128 && groups % chosen.splits == 0 ? PLAN_SLICES_TILE256 : PLAN_SLICES_SHORT_A;
    }
  } else if (aligned && nblk * nbatch < n_cu) { // (8-bit operands: smaller tiles in one pass are the only alternative here)
    chosen = choose(true, INT64_MAX);
    if (want && chosen.splits > 1)
      *optional = choose(false, INT64_MAX).splits == 1;
  }
  if (chosen.splits > 1) {
    if (want)
      *want = (int64_t)chosen.splits * p.M * p.N;
    // less workspace than that: what is best with what there is; of a caller's slices fewer, or none
    if (p.cfg_tile == 0 && (int64_t)chosen.splits * p.M * p.N > ws_cap)
      chosen = choose(true, ws_cap);
    while (chosen.splits > 1 &&
           ((int64_t)chosen.splits * p.M * p.N > ws_cap || (chosen.plan == PLAN_SLICES_TILE256 && groups % chosen.splits != 0)))
      chosen.splits--;
    if (chosen.splits == 1 && p.cfg_tile != 0)
      chosen.plan = PLAN_TILE256;
  }
  const int plan = chosen.plan, splits = chosen.splits, rows128 = chosen.rows128;
  const int64_t nblk128 = ((p.M + rows128 - 1) / rows128) * ((p.N + 127) / 128);
  if (want && !cfg)
    return 0;
  if (splits > 1) {
    const bool by128 = plan == PLAN_SLICES_TILE128, by256 = plan == PLAN_SLICES_TILE256;
    const int tiles = (int)(by128 ? nblk128 : nblk);
    c.kernel = GK_SPLITK, c.split_k = splits, c.workgroups = tiles * splits;
    if (by128) {
      c.bm = rows128, c.bn = 128, c.kbytes = T128_KB, c.stages = tile128_stages<ES>(rows128, 128, p.K, p.trans_b, splits, nblk128 * splits);
      c.waves_m = c.waves_n = 2, c.wave_m = rows128 / 2, c.wave_n = 64, c.mfma_m = c.mfma_n = 16, c.mfma_k = 32;
    } else if (by256) {
      c.kbytes = 64, c.stages = 4, c.waves_m = 2, c.waves_n = 2, c.wave_m = 128, c.wave_n = 128;
      c.mfma_m = c.mfma_n = 16, c.mfma_k = 64 / ES;
    } else {
      c.kbytes = FastGemm<ES, G_FAST_KS, G_FAST_WJ, true>::KB, c.stages = FastGemm<ES, G_FAST_KS, G_FAST_WJ, true>::NST;
      c.waves_m = 2, c.waves_n = 8 / G_FAST_WJ, c.wave_m = 128, c.wave_n = 32 * G_FAST_WJ;
      c.mfma_m = c.mfma_n = 32, c.mfma_k = 32 / ES;
    }
    if (cfg)
      *cfg = c;
    if (dry)
      return 0;
    p.splits = splits;
    p.partial = ws;
    if constexpr (ES == 2) {
      if (by128) { // the kernel cuts K itself: blockIdx.y = slice
        const int rc = gcmi_launch_tile128(&p, ES, rows128, 128, (unsigned)tiles, (unsigned)splits, stream);
        if (rc)
          return rc;
      } else if (by256) { // equal slices as a strided batch with f32 results
        GemmParams q = p;
        q.K = p.K / splits, q.batch = splits;
        q.a_bs = q.K, q.b_bs = p.trans_b ? q.K : q.K * p.ldb, q.c_bs = p.M * p.N;
        q.C = ws, q.ldc = p.N, q.out_dt = DT_F32;
        q.bias = nullptr, q.act = ACT_NONE, q.residual = nullptr, q.partial = nullptr, q.splits = 0;
        const dim3 grid((unsigned)tiles, (unsigned)splits);
        if (p.trans_b)
          hipLaunchKernelGGL((gemm_tile256_w4_kernel<ES, true>), grid, dim3(256), 0, stream, q);
        else
          hipLaunchKernelGGL(gemm_tile256_w4_kernel<ES>, grid, dim3(256), 0, stream, q);
      } else if (p.trans_b)
        hipLaunchKernelGGL((gemm_tile256_fast_kernel<ES, G_FAST_KS, G_FAST_WJ, true, true>),
                           dim3((unsigned)(tiles * splits)), dim3(1024 / G_FAST_WJ), 0, stream, p);
      else
        hipLaunchKernelGGL((gemm_tile256_fast_kernel<ES, G_FAST_KS, G_FAST_WJ, true>), dim3((unsigned)(tiles * splits)),
                           dim3(1024 / G_FAST_WJ), 0, stream, p);
    }
    launch_splitk_reduce(p, stream);
    return hipGetLastError() == hipSuccess ? 0 : 5;
  }
  if (plan == PLAN_TILE128) {
    c.kernel = GK_TILE128, c.bm = rows128, c.bn = 128, c.kbytes = T128_KB;
    c.stages = tile128_stages<ES>(rows128, 128, p.K, p.trans_b, 1, nblk128 * nbatch);
    c.waves_m = c.waves_n = 2, c.wave_m = rows128 / 2, c.wave_n = 64, c.mfma_m = c.mfma_n = 16, c.mfma_k = 64 / ES;
    c.workgroups = (int32_t)nblk128;
    if (cfg)
      *cfg = c;
    if (dry)
      return 0;
    return gcmi_launch_tile128(&p, ES, rows128, 128, (unsigned)nblk128, (unsigned)nbatch, stream);
  }
  // Whole tiles: 4 waves of 128 x 128 unless the caller asks for 8 waves of 128 x 64.  Results of 8-bit operands
  // leave the 4-wave kernel as bf16, f32 or as the raw s32 accumulators (same main loop, the epilogue is a plain
  // store).  Tiles that stick out of C and a K that ends inside a ring group (`ragged`): the 4-wave kernel.  Anything
  // else (a K or N of no whole 16-byte chunks, unaligned rows): the bounds-checked kernel.
  const bool w4_can = fast || ragged;
  const bool use_w4 = w4_can && (p.cfg_waves != 8 || !fast);
  const bool tiled = fast || use_w4; // one of the kernels with the LDS ring
  c.kernel = !tiled ? GK_EDGE : (use_w4 ? GK_WAVES4 : GK_WAVES8);
  c.kbytes = tiled ? 64 : G_KBYTES, c.stages = tiled ? 4 : 2;
  c.waves_m = 2, c.waves_n = use_w4 ? 2 : 4, c.wave_m = 128, c.wave_n = use_w4 ? 128 : 64;
  c.mfma_m = c.mfma_n = tiled ? 16 : 32, c.mfma_k = (tiled ? 64 : 32) / ES;
  // More than a round of whole tiles with a poorly filled last round: the tiles of the last round are a block of
  // columns (or rows) of C; where 128 x 128 tiles are estimated to finish that block clearly sooner than the large
  // ones (up to about 40 % of a round), it becomes a launch of its own behind the whole rounds.  Both kernels add
  // the products of an element in the same order, so C has the same bits either way.
  int64_t tail_cols = 0, tail_rows = 0;
  if (use_w4 && fast && nbatch == 1 && p.cfg_tile == 0 && t128_can && nblk > n_cu && nblk % n_cu != 0) {
    const int64_t tail = nblk % n_cu;
    const double t256 = GCMI_US_FIXED_256 + gcmi_us_per_group_256((double)tail / n_cu) * groups;
    const double t128 = GCMI_US_FIXED_128 + 2.0 + gcmi_us_per_group_128(4.0 * tail / n_cu) * groups * (double)((4 * tail + 2 * n_cu - 1) / (2 * n_cu));
    if (t128 < GCMI_ONE_PASS_MARGIN * t256) {
      if (tail % tiles_m == 0)
        tail_cols = tail / tiles_m * G_BN;
      else if (tail % tiles_n == 0)
        tail_rows = tail / tiles_n * G_BM;
    }
  }
  if (tail_cols || tail_rows)
    c.workgroups = (int32_t)(nblk - nblk % n_cu + 4 * (nblk % n_cu));
  // Large tiles that leave much of a round idle: another tile where it is estimated clearly ahead, in one pass, the same bits
  // (same products in the same order, same epilogue).  The 184 sizes of the estimates gain 1.10 on the average (the best tile of
  // each would give 1.118), two lose more than 2 % (at most 5 %).  us, 256 x 256 / chosen: 1000 x 11008, K 4096 82.2 / 73.9 on 256 x 192;
  // 2655 x 3520, K 3800 73.6 / 64.9 likewise; 1643 x 10048, K 1408 (280 tiles) 66.5 / 57.5 on 192 x 128; 3597 x 4672, K 128 22.0 / 15.6
  // on 128 x 128.  Under half a round (the estimates above decide) and past three the sizes were not measured.  Past one, a K of 4096 and
  // more was not fitted either and keeps the large tile, which is no line by speed: 2048 x 11008 165.8 there, 143.7 on 256 x 192, 4096 x
  // 11008 263.7 / 283.0.
  if (ES == 2 && use_w4 && t128_can && !tail_cols && !tail_rows && p.cfg_tile == 0 && !p.cfg_waves && !p.cfg_split_k &&
      2 * nblk * nbatch >= n_cu && nblk * nbatch < (p.K < 4096 ? 3 : 1) * n_cu) {
    const GemmTileCost *tile = &GCMI_TILE_COSTS[0];
    double best = 0.95 * gcmi_us_tile(*tile, p.M, p.N, nbatch, groups, n_cu);
    for (const GemmTileCost &t : GCMI_TILE_COSTS) {
      const double us = gcmi_us_tile(t, p.M, p.N, nbatch, groups, n_cu);
      if (us < best)
        best = us, tile = &t;
    }
    if (tile->rows != 256 || tile->cols != 256) {
      const int64_t tiles = ((p.M + tile->rows - 1) / tile->rows) * ((p.N + tile->cols - 1) / tile->cols);
      c.kernel = GK_TILE128, c.bm = tile->rows, c.bn = tile->cols, c.wave_m = tile->rows / 2, c.wave_n = tile->cols / 2;
      c.workgroups = (int32_t)tiles, c.stages = tile128_stages<ES>(tile->rows, tile->cols, p.K, p.trans_b, 1, tiles * nbatch);
      if (cfg)
        *cfg = c;
      if (dry)
        return 0;
      return gcmi_launch_tile128(&p, ES, tile->rows, tile->cols, (unsigned)tiles, (unsigned)nbatch, stream);
    }
  }
  if (cfg)
    *cfg = c;
  if (dry)
    return 0;
  if (tail_cols || tail_rows) {
    GemmParams head = p, rest = p;
    const int bias_es = p.bias_dt == DT_BF16 ? 2 : 4;
    if (tail_cols) {
      const int64_t n1 = p.N - tail_cols;
      head.N = n1, rest.N = tail_cols;
      rest.B = reinterpret_cast<const char *>(p.B) + (p.trans_b ? n1 * p.ldb : n1) * ES;
      rest.C = reinterpret_cast<char *>(p.C) + n1 * out_es;
      if (p.bias)
        rest.bias = reinterpret_cast<const char *>(p.bias) + n1 * bias_es;
      if (p.scale)
        rest.scale = p.scale + n1;
      if (p.colsum)
        rest.colsum = p.colsum + n1;
      if (p.residual)
        rest.residual = reinterpret_cast<const char *>(p.residual) + n1 * res_es;
    } else {
      const int64_t m1 = p.M - tail_rows;
      head.M = m1, rest.M = tail_rows;
      rest.A = reinterpret_cast<const char *>(p.A) + m1 * p.lda * ES;
      rest.C = reinterpret_cast<char *>(p.C) + m1 * p.ldc * out_es;
      if (p.residual)
        rest.residual = reinterpret_cast<const char *>(p.residual) + m1 * p.ldr * res_es;
    }
    const dim3 hgrid((unsigned)(nblk - nblk % n_cu));
    if (p.trans_b) {
      if constexpr (ES == 2) {
        hipLaunchKernelGGL((gemm_tile256_w4_kernel<ES, true>), hgrid, dim3(256), 0, stream, head);
      }
    } else {
      hipLaunchKernelGGL(gemm_tile256_w4_kernel<ES>, hgrid, dim3(256), 0, stream, head);
    }
    return gcmi_launch_tile128(&rest, ES, 128, 128, (unsigned)(4 * (nblk % n_cu)), 1, stream);
  }
  dim3 grid((unsigned)nblk, (unsigned)nbatch), block(G_THREADS);
  if (use_w4) {
    if constexpr (ES == 2) {
      if (p.trans_b) {
        hipLaunchKernelGGL((gemm_tile256_w4_kernel<ES, true>), grid, dim3(256), 0, stream, p);
        return hipGetLastError() == hipSuccess ? 0 : 5;
      }
    }
    hipLaunchKernelGGL(gemm_tile256_w4_kernel<ES>, grid, dim3(256), 0, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : 5;
  }
  if constexpr (ES == 2) {
    if (p.trans_b) {
      if (fast)
        hipLaunchKernelGGL((gemm_tile256_mi16_kernel<ES, true>), grid, dim3(512), 0, stream, p);
      else
        hipLaunchKernelGGL((gemm_tile256_kernel<ES, true, true>), grid, block, 0, stream, p);
      return hipGetLastError() == hipSuccess ? 0 : 5;
    }
  }
  if (fast)
    hipLaunchKernelGGL(gemm_tile256_mi16_kernel<ES>, grid, dim3(512), 0, stream, p);
  else
    hipLaunchKernelGGL((gemm_tile256_kernel<ES, true>), grid, block, 0, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

} // namespace gcmi
