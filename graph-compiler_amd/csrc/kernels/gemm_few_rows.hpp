// GEMMs of few rows of A (up to 256; 2048 of 8 bits) against weights that are no stream worth slicing: bf16 x bf16 with weights
// stored [K,N] or [N,K], and 8-bit x s8 with weights stored [K,N], alone or in a strided batch.  C[M,N] = epilogue(A . W) in
// ONE launch.
// What bounds such a call is the way launch -> loads -> sums -> store, once: the tile kernels' workgroup walks all of K
// through one ring behind barriers (a 256 x 256 tile takes 60 us for 2 x 5456, K 3264, on 22 compute units), and K slices
// over workgroups cost a second launch.  Here K is cut over the waves of a workgroup:
//   * a workgroup has 16 * NT columns and 16 * MT rows; wave w takes stages w, w + W, ... of 128 bytes of K per row, each
//     into an LDS ring of its own by global_load_lds_dwordx4, D stages deep: no barrier and no wait for another wave until
//     the W partial sums are added (ascending, a fixed order: results do not depend on timing).  The waves' stages lie
//     beside each other in memory, so eight of them read runs of 1 KiB of every row.  (Deeper rings, sixteen waves or stages
//     of 64 bytes: no difference to 5 % slower; it is the number of lines a compute unit looks up that counts.)
//   * the smallest tile that fits the GPU in one round, so that as many compute units as there are pull on the weights.  A
//     run of neighbouring tiles goes to one XCD, whose L2 reads a line of [K,N] weights once for all of them (with the
//     tiles dealt out over the XCDs, 8-bit 30 x 4960, K 3232 took 24.3 us, 9.2 now; 30 x 11008, K 4096 19.3 and 12.4).
//   * rows of 128 bytes (A, [N,K] weights) lie at chunk ^ row % 8; k-rows of [K,N] weights are read through the transposing
//     LDS loads, at a chunk that spreads them over the banks.
// The columns' bias, scale and column sums are fetched before the loop by the wave that finishes them.
// The k that a wave owns and the order of the sums depend on M, N and the size of the batch only: both layouts of the weights
// give the same bits.
// Measured, us per call, graph-replayed over 64 MB of weights: bf16 [N,K] 3 x 1712, K 2736 48 -> 6; 19 x 1648, K 3592 63.4 ->
// 7.7; 13 x 1792, K 1856 8.4 (two launches) -> 5.0; [K,N] 10 x 320, K 3200 53 -> 8.5; 8-bit 10 x 512, K 3776 36 -> 7.7; 32 x
// 11008, K 4096 20.0 -> 12.5 (3.7 TB/s of weights).
#pragma once
#include "gemm_tile256.hpp"

namespace gcmi {

template <int ES, bool TB, int MT, int NT, int W, int D> struct FewRows {
  static constexpr int STEPS = 2, KB = 64 * STEPS, BK = KB / ES; // MFMA steps, bytes and elements of K per stage
  static constexpr int A_BYTES = 16 * MT * KB, STAGE = A_BYTES + 16 * NT * KB;
  static constexpr int NA = STEPS * MT, NB = STEPS * NT, PER = NA + NB; // requests per stage: 1 KiB each
  static constexpr int RING = D * STAGE, SMEM = W * RING;
  static constexpr int BROW = 16 * NT * ES;                   // bytes of a k-row of [K,N] weights
  static_assert(W * MT * NT * 1024 <= SMEM, "the partial sums lie over the rings");
  static_assert(D * PER <= 63, "requests in flight are counted in six bits");
  static_assert(W % NT == 0, "a wave finishes tiles of one column group");
  // where the 16-byte chunk of a row of KB bytes lies inside it (rows 16 apart alike)
  static __device__ __forceinline__ int row_swz(int row) { return row & 7; }
  // where the 16-byte chunk of a k-row lies inside it
  static __device__ __forceinline__ int swz(int krow) {
    if constexpr (ES == 2 && NT == 4) // 8 chunks; a transposing read takes 4 k-rows per 16 lanes, 8 apart
      return (((krow >> 1) & 1) | (((krow >> 3) & 1) << 1)) << 1;
    else if constexpr (ES == 1 && NT == 4) // 4 chunks; 8 k-rows per 16 lanes, 16 apart
      return ((krow >> 2) & 1) | (((krow >> 4) & 1) << 1);
    else
      return 0;
  }
};

// one row quad of an 8-bit product: the 4-wave tile kernels' epilogue
template <bool TAME>
__device__ __forceinline__ void few_rows_store_int8(const GemmParams &p, const i32x4_t &c, int64_t m, int64_t n, const f32x4_t &bias4,
                                                    const f32x4_t &scale4, const i32x4_t &cs4) {
#define GCMI_FEW_CASE(ACT, OUT, K)                                                                                    \
  case (int)ACT + 8 * K:                                                                                              \
    w4_epilogue_row<1, ACT, OUT, false, false, false, TAME>(p, c, m, n, bias4, scale4, cs4);                          \
    break;
  const int out_kind = p.out_dt == DT_BF16 ? 0 : (p.out_dt == DT_S32 ? 2 : 1);
  switch ((out_kind == 2 ? (int)ACT_NONE : p.act) + 8 * out_kind) {
    GCMI_FEW_CASE(ACT_RELU, DT_BF16, 0)
    GCMI_FEW_CASE(ACT_GELU_ERF, DT_BF16, 0)
    GCMI_FEW_CASE(ACT_GELU_TANH, DT_BF16, 0)
    GCMI_FEW_CASE(ACT_SIGMOID, DT_BF16, 0)
    GCMI_FEW_CASE(ACT_NONE, DT_F32, 1)
    GCMI_FEW_CASE(ACT_RELU, DT_F32, 1)
    GCMI_FEW_CASE(ACT_GELU_ERF, DT_F32, 1)
    GCMI_FEW_CASE(ACT_GELU_TANH, DT_F32, 1)
    GCMI_FEW_CASE(ACT_SIGMOID, DT_F32, 1)
    GCMI_FEW_CASE(ACT_NONE, DT_S32, 2)
  default:
    w4_epilogue_row<1, ACT_NONE, DT_BF16, false, false, false, TAME>(p, c, m, n, bias4, scale4, cs4);
    break;
  }
#undef GCMI_FEW_CASE
}

template <int ES, bool TB, int MT, int NT, int W, int D> __global__ __launch_bounds__(64 * W) void gemm_few_rows_kernel(GemmParams p) {
  static_assert(!TB || ES == 2, "weights stored [N,K]: bf16 only");
  typedef FewRows<ES, TB, MT, NT, W, D> F;
  constexpr int STEPS = F::STEPS;
  typedef typename std::conditional<ES == 2, f32x4_t, i32x4_t>::type acc4_t;
  __shared__ __align__(1024) char smem[F::SMEM];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r16 = lane & 15, g16 = lane >> 4;
  const int tiles_m = (int)((p.M + 16 * MT - 1) / (16 * MT)), tiles_n = (int)((p.N + 16 * NT - 1) / (16 * NT));
  // workgroup i runs on XCD i % 8: each XCD walks its own run of panels (the grid is rounded up to whole runs), through the
  // matrices of a batch one after the other: with a grid of their own, rounded up each, 84 matrices of three tiles met on
  // three XCDs (84 x 46 x 176, K 960 25 us, 12 in one run)
  const int tile = (int)(blockIdx.x & 7) * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3), tm = tile % tiles_m;
  int tn = tile / tiles_m, bz = 0; // bz: strided batch
  if (p.batch > 1)
    bz = tn / tiles_n, tn -= bz * tiles_n;
  if (tn >= tiles_n || (p.batch > 1 && bz >= p.batch))
    return;
  const int64_t m0 = (int64_t)tm * 16 * MT, n0 = (int64_t)tn * 16 * NT;
  const int rows_in = (int)min((int64_t)16 * MT, p.M - m0), cols_in = (int)min((int64_t)16 * NT, p.N - n0);
  p.A = reinterpret_cast<const char *>(p.A) + bz * p.a_bs * ES;
  p.B = reinterpret_cast<const char *>(p.B) + bz * p.b_bs * ES;
  p.C = reinterpret_cast<char *>(p.C) + bz * p.c_bs * (p.out_dt == DT_BF16 ? 2 : 4);
  if (ES == 2 && p.residual)
    p.residual = reinterpret_cast<const char *>(p.residual) + bz * p.c_bs * (p.residual_dt == DT_BF16 ? 2 : 4);
  const int64_t lda_b = p.lda * ES, ldb_b = p.ldb * ES;

  // what belongs to the columns that this wave finishes, as it lies in memory (looked at behind the loop)
  typedef uint16_t u16x4u_t __attribute__((ext_vector_type(4), aligned(2)));
  typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));
  typedef int i32x4u_t __attribute__((ext_vector_type(4), aligned(4)));
  const int64_t nw = n0 + 16 * (wave % NT) + 4 * g16;
  const bool finishes = wave < MT * NT && nw < p.N; // N is a multiple of 4
  u16x4u_t bias16 = {0, 0, 0, 0};
  f32x4u_t bias32 = {0.f, 0.f, 0.f, 0.f}, scale4 = {1.f, 1.f, 1.f, 1.f};
  i32x4u_t sums4 = {0, 0, 0, 0};
  if (finishes) {
    if (p.bias && p.bias_dt == DT_BF16)
      bias16 = *reinterpret_cast<const u16x4u_t *>(reinterpret_cast<const uint16_t *>(p.bias) + nw);
    if (p.bias && p.bias_dt != DT_BF16)
      bias32 = *reinterpret_cast<const f32x4u_t *>(reinterpret_cast<const float *>(p.bias) + nw);
    if (ES == 1 && p.scale)
      scale4 = *reinterpret_cast<const f32x4u_t *>(p.scale + nw);
    if (ES == 1 && p.colsum)
      sums4 = *reinterpret_cast<const i32x4u_t *>(p.colsum + nw);
  }

  const int stages = (int)((p.K + F::BK - 1) / F::BK), n_st = (stages - wave + W - 1) / W; // this wave's
  const int k_end = (int)(p.K - (int64_t)(stages - 1) * F::BK);                            // elements of the last stage
  // requests: 8 rows of 128 bytes, or 1024 / BROW k-rows.  Rows, chunks and k-rows outside read the last ones inside.
  uint32_t a_src[F::NA], b_src[F::NB];
  auto offsets = [&](int k_in) {
    constexpr int CPR = F::KB / 16, RPR = 64 / CPR; // chunks of a row, rows of a request
    const int chunks = k_in * ES / 16, row = lane / CPR, c = min((lane % CPR) ^ F::row_swz(row), chunks - 1);
#pragma unroll
    for (int i = 0; i < F::NA; i++)
      a_src[i] = (uint32_t)(min(RPR * i + row, rows_in - 1) * lda_b + c * 16);
#pragma unroll
    for (int i = 0; i < F::NB; i++) {
      if constexpr (TB) {
        b_src[i] = (uint32_t)(min(RPR * i + row, cols_in - 1) * ldb_b + c * 16);
      } else {
        constexpr int CPR = F::BROW / 16; // chunks of a k-row
        const int krow = i * (64 / CPR) + lane / CPR, cb = (lane % CPR) ^ F::swz(krow);
        b_src[i] = (uint32_t)(min(krow, k_in - 1) * ldb_b + min(cb, cols_in * ES / 16 - 1) * 16);
      }
    }
  };
  const int64_t b_step = TB ? (int64_t)F::KB : (int64_t)F::BK * ldb_b;
  const char *a_ptr = reinterpret_cast<const char *>(p.A) + m0 * lda_b + (int64_t)wave * F::KB;
  const char *b_ptr = reinterpret_cast<const char *>(p.B) + (TB ? n0 * ldb_b : n0 * ES) + wave * b_step;
  char *const ring = smem + wave * F::RING;
  // (written as assembly: of requests that the compiler knows it awaits all in flight before every read of LDS)
  const uint32_t ring_at = (uint32_t)(uintptr_t)(GCMI_LDS char *)ring;
  auto request = [&](const char *base, uint32_t off, uint32_t at) { // 16 bytes per lane from base + off to LDS at + 16 * lane
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(off), "s"(base), "s"(at) : "m0", "memory");
  };
  auto issue = [&](int st, int i) { // this wave's stage i, to the slot at st
    if (wave + i * W == stages - 1)
      offsets(k_end);
    const char *a = a_ptr + (int64_t)i * (W * F::KB), *b = b_ptr + i * (W * b_step);
#pragma unroll
    for (int r = 0; r < F::NA; r++)
      request(a, a_src[r], ring_at + st + r * 1024);
#pragma unroll
    for (int r = 0; r < F::NB; r++)
      request(b, b_src[r], ring_at + st + F::A_BYTES + r * 1024);
  };
  acc4_t acc[NT][MT]; // rows 16 * it + lane % 16, columns 16 * jt + 4 * (lane / 16) .. + 3 (weights as first operand)
#pragma unroll
  for (int jt = 0; jt < NT; jt++)
#pragma unroll
    for (int it = 0; it < MT; it++)
      acc[jt][it] = acc4_t{0, 0, 0, 0};
  uint4 fa[STEPS][MT], fb[STEPS][NT];
  auto read = [&](const char *st) {
#pragma unroll
    for (int u = 0; u < STEPS; u++) {
      const int at = r16 * F::KB + (((4 * u + g16) ^ F::row_swz(r16)) << 4);
#pragma unroll
      for (int it = 0; it < MT; it++)
        fa[u][it] = *reinterpret_cast<const uint4 *>(st + at + it * 16 * F::KB);
#pragma unroll
      for (int jt = 0; jt < NT; jt++) {
        if constexpr (TB) {
          fb[u][jt] = *reinterpret_cast<const uint4 *>(st + F::A_BYTES + at + jt * 16 * F::KB);
        } else {
          // the 16 lanes of a group hand the transposing read RG k-rows x 16 columns in 8-byte pieces
          constexpr int RG = ES == 2 ? 4 : 8;
          const int kk = ES == 2 ? r16 >> 2 : r16 >> 1, cc = ES == 2 ? r16 & 3 : r16 & 1;
          const int chunk = ES == 2 ? 2 * jt + (cc >> 1) : jt, sub = ES == 2 ? (cc & 1) * 8 : cc * 8;
          const int krow = (64 / ES) * u + 2 * RG * g16 + kk;
          const char *q = st + F::A_BYTES + sub;
          const uint2 lo = MfmaOp<ES>::tr_read(q + krow * F::BROW + ((chunk ^ F::swz(krow)) << 4));
          const uint2 hi = MfmaOp<ES>::tr_read(q + (krow + RG) * F::BROW + ((chunk ^ F::swz(krow + RG)) << 4));
          fb[u][jt] = make_uint4(lo.x, lo.y, hi.x, hi.y);
        }
      }
    }
  };
  const uint32_t a_xor = p.a_xor;
  auto products = [&]() {
#pragma unroll
    for (int u = 0; u < STEPS; u++)
#pragma unroll
      for (int it = 0; it < MT; it++) {
        if constexpr (ES == 2) {
#pragma unroll
          for (int jt = 0; jt < NT; jt++)
            acc[jt][it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, fb[u][jt]),
                                                                  __builtin_bit_cast(bf16x8_t, fa[u][it]), acc[jt][it], 0, 0, 0);
        } else {
          const uint4 f = make_uint4(fa[u][it].x ^ a_xor, fa[u][it].y ^ a_xor, fa[u][it].z ^ a_xor, fa[u][it].w ^ a_xor);
#pragma unroll
          for (int jt = 0; jt < NT; jt++)
            acc[jt][it] = __builtin_amdgcn_mfma_i32_16x16x64_i8(__builtin_bit_cast(i32x4_t, fb[u][jt]), __builtin_bit_cast(i32x4_t, f),
                                                                acc[jt][it], 0, 0, 0);
        }
      }
  };
  // what lies behind K in the last stage: zeros in the weights, and for bf16 in A (an infinity times zero would be a NaN;
  // 8-bit bytes of A are any byte)
  auto cut = [&]() {
#pragma unroll
    for (int u = 0; u < STEPS; u++)
      if ((4 * u + g16) * (16 / ES) >= k_end) {
#pragma unroll
        for (int jt = 0; jt < NT; jt++)
          fb[u][jt] = make_uint4(0, 0, 0, 0);
        if constexpr (ES == 2)
#pragma unroll
          for (int it = 0; it < MT; it++)
            fa[u][it] = make_uint4(0, 0, 0, 0);
      }
  };
  offsets(F::BK);
#pragma unroll
  for (int d = 0; d < D; d++)
    if (d < n_st)
      issue(d * F::STAGE, d);
  int slot = 0;
  for (int i = 0; i < n_st; i++) {
    // stage i has landed (the D - 1 behind it may be in flight; near the end fewer were asked for and all are awaited)
    if (i + D - 1 < n_st)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((D - 1) * F::PER) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const int st = slot * F::STAGE;
    read(ring + st);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // the reads are over: the slot is free
    if (i + D < n_st)
      issue(st, i + D);
    if (k_end < F::BK && wave + i * W == stages - 1)
      cut();
    products();
    slot = slot + 1 < D ? slot + 1 : 0;
  }
  // the waves' sums, in ascending order; a wave finishes every W-th tile
  __syncthreads();
  acc4_t *red = reinterpret_cast<acc4_t *>(smem);
#pragma unroll
  for (int it = 0; it < MT; it++)
#pragma unroll
    for (int jt = 0; jt < NT; jt++)
      red[(wave * MT * NT + it * NT + jt) * 64 + lane] = acc[jt][it];
  __syncthreads();
  f32x4_t bias4;
  i32x4_t cs4;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    bias4[e] = !p.bias ? -0.0f : p.bias_dt == DT_BF16 ? bf16_bits_to_f32(bias16[e]) : bias32[e]; // absent: nothing is added, not even to -0.0
    cs4[e] = p.comp * sums4[e];
  }
  bool tame = ES == 1; // see w4_epilogue_half
#pragma unroll
  for (int e = 0; e < 4; e++)
    tame = tame && fabsf(scale4[e]) < 0x1p90f && fabsf(bias4[e]) < 0x1p120f;
#pragma unroll 1
  for (int t = wave; t < MT * NT; t += W) {
    acc4_t v = red[t * 64 + lane];
#pragma unroll
    for (int w = 1; w < W; w++) {
      const acc4_t o = red[(w * MT * NT + t) * 64 + lane];
#pragma unroll
      for (int e = 0; e < 4; e++)
        v[e] += o[e];
    }
    const int64_t m = m0 + 16 * (t / NT) + r16;
    if (m >= p.M || !finishes)
      continue;
    if constexpr (ES == 2)
      epilogue_store4(p, v, m, nw, bias4);
    else if (tame)
      few_rows_store_int8<true>(p, v, m, nw, bias4, scale4, cs4);
    else
      few_rows_store_int8<false>(p, v, m, nw, bias4, scale4, cs4);
  }
}

// The tile: 16 * mt rows and 16 * nt columns per workgroup.  A workgroup's time is that of its operands (about 45 KB a us
// past 3 us), so the tile with the fewest of them wins that needs no second round of workgroups; a second round costs a
// workgroup's time again.
struct FewRowsTile {
  int mt, nt, waves, stages; // waves that share K, stages of a wave's ring
  int64_t blocks, rounds;
};
static FewRowsTile few_rows_tile(int64_t M, int64_t N, int64_t nbatch) {
  const int64_t n_cu = gcmi_num_cus();
  FewRowsTile best{};
  int64_t best_cost = INT64_MAX;
  for (int mt = 4; mt >= 1; mt /= 2) // (of equal tiles the one with more rows: the weights are read by fewer workgroups)
    for (int nt = 1; nt <= 4; nt *= 2) {
      const int64_t blocks = ((M + 16 * mt - 1) / (16 * mt)) * ((N + 16 * nt - 1) / (16 * nt)), rounds = (blocks * nbatch + n_cu - 1) / n_cu;
      const int64_t cost = rounds * (mt + nt);
      if (cost < best_cost || (cost == best_cost && blocks < best.blocks)) {
        const int waves = nt == 1 && mt < 4 ? 8 : 4;
        best = {mt, nt, waves, waves == 8 || mt + nt == 8 ? 2 : 3, blocks, rounds};
        best_cost = cost;
      }
    }
  return best;
}

// Where this kernel is the faster one, measured over 1 to 256 rows, 64 to 11008 columns and K 64 to 4096 (us, graph-replayed,
// the other kernel / this):
//   * bf16 below 32 rows, where the others walk K in one workgroup per 256 columns or slice it: 3 x 1712, K 2736 48 / 6;
//     10 x 640, K 3968 8.0 / 5.6.  Wide weights (4 Mi and more of them, K in whole groups of 128) stream (gemm_rows32.hpp).
//   * more rows while one round of workgroups, or two of small ones with 8-bit operands, holds them (rounds * (mt + nt)): 83 x
//     768, K 3136 12.0 / 8.5; 8-bit 83 x 768, K 3136 18.8 / 8.5; 80 x 10384, K 1072 13.3 / 12.1; past that 128 x 128 tiles
//     re-read the operands less often (8-bit 234 x 10816, K 3584 23.5 / 31.8; bf16 150 x 5736, K 512 8.9 / 10.8).
//     The largest tiles with a bf16 K of 256 or less, or of up to four whole groups, leave a wave two stages at most: 177 x 3328,
//     K 256 6.8 / 7.8; 112 x 7072, K 384 8.1 / 8.8; 10 matrices of 189 x 448, K 256 6.4 / 7.6; with a longer K or a tail 92
//     random sizes 1.0 to 1.3 times (96 x 7032, K 616 12.5 / 10.0).
//   * 8-bit operands, for which the tile kernels have no K slices, up to 2048 rows while one round holds them: 45 random sizes
//     of 257 to 2000 rows 1.75 times on the average (679 x 608, K 3568 23.6 / 11.1; 1328 x 768, K 976 11.0 / 8.1).  In two rounds
//     128 x 128 tiles are level or ahead up to a cost of 16 (562 x 2480, K 5184 32.4 / 34.3; 607 x 2976, K 25168 129 / 124), past it
//     ahead (968 x 2128, K 4288 25.7 / 42.1).  The ends at 512 columns, K 4096 and 2048 rows are no lines by speed: 180 random sizes
//     past them in one round, 16 to 2600 columns, K to 30000, 19000 rows, are 1.1 to 4.8 times ahead here too (257 x 1024, K 4112
//     21.4 / 11.6; 257 x 496, K 2048 14.0 / 7.0; 1503 x 560, K 26368 117 / 71).
//   * with a K that ends inside a group of 128 nothing streams, so these are taken whatever the weights' size, 32 rows (32 x 4096,
//     K 1376 12.3 / 8.0, 32 x 6336, K 2136 14.4 / 10.4) and 129 to 256 (140 x 264, K 1048 9.8 / 5.5, 169 x 2400, K 1464 14.7 /
//     10.0, 248 x 2656, K 776 13.3 / 10.5) like those between: 100 random sizes of them 1.5 times with [K,N] weights, 1.65 with
//     [N,K]; a long K see below.
//   * a K of 272 bytes or less is the tile kernels', which is no line by speed: this one would be ahead there as well, up to 31
//     rows 9 to 14 us / 3 to 7, from 32 on 5.0 to 7.2 / 3.0 to 5.4 up to a cost of 6 (8-bit 8); at a bf16 cost of 8 5.7 / 6.9.
template <int ES> static bool few_rows_wanted(const GemmParams &p, const FewRowsTile &t) {
  const int64_t cost = t.rounds * (t.mt + t.nt);
  if (p.K * ES <= 272 || (p.M >= 32 && cost > (ES == 2 ? 8 : 12)))
    return false;
  if (ES == 2 && p.M >= 32 && cost > 6 && (p.K <= 256 || (p.K <= 512 && p.K % 128 == 0)))
    return false;
  if (p.M > 256) // 8-bit operands
    return t.rounds == 1 && p.N >= 512 && p.K <= 4096;
  if (ES == 1 || p.M < 32)
    return true;
  return p.K % 128 != 0 || p.N * p.K < (int64_t)1 << 22;
}

// A wave walks its share of K alone, a stage in about 0.85 us ([K,N]; 0.4 where N is no more than 40) or 0.35 ([N,K]; half as much
// again with rows that are no whole lines), up to 1.3 on the larger tiles, while K slices over workgroups take their 10 to 15 us
// and little more for a longer K.  So past a K they win, where another kernel has them.  Measured over 32 to 256 rows of 16 to
// 8192 columns (530 random sizes from the cache, 440, K 1000 to 14000, from memory too: m), by the sixteenths of rows and
// columns of a tile, us, slices / this:
//   [K,N] 2   112 x 528, K 5824 14.6 / 12.5   32 x 168, K 5968 12.8 / 14.2   169 x 168, K 7776 13.7 / 16.0  48 x 112, K 188208 37 / 302
//         2, few columns   157 x 40, K 8704 14.4 / 11.9   143 x 16, K 13696 17.4 / 11.8   46 x 24, K 26112 25 / 23   256 x 32, K 24448 18 / 25
//         3   74 x 1488, K 4552 14.6 / 12.6 (m 16.2 / 16.4)   32 x 3840, K 4920 15.4 / 16.7 (m 16.6 / 24.1)   49 x 1880, K 5104 14.8 / 14.4 (m 15.5 / 17.7)
//         4   100 x 1928, K 4320 15.9 / 15.8 (m 18.2 / 17.1)   55 x 2136, K 4744 15.1 / 16.4 (m 15.7 / 21.0)
//         5   41 x 4400, K 3192 15.9 / 13.5 (m 16.7 / 17.4)   104 x 2200, K 5056 17.7 / 18.4 (m 18.6 / 23.0)
//         6   119 x 2216, K 3136 16.0 / 14.0 (m 19.3 / 17.4)   206 x 1536, K 4304 16.4 / 15.7 (m 17.7 / 21.5)   102 x 2808, K 4600 17.7 / 19.0 (m 20.6 / 24.3)
//         6, full   37 x 7432, K 5344 25.1 / 21.9 (m 26.1 / 26.5)   40 x 7984, K 5720 27.2 / 24.1 (m 28.2 / 32.2)   56 x 7176, K 5512 25.5 / 26.2 (m 27.0 / 30.5)
//         8   134 x 4112, K 3888 25.1 / 23.4 (m 25.3 / 24.4)   100 x 6208, K 3744 18.7 / 19.2 (m 21.3 / 23.8)   79 x 6216, K 4312 21.6 / 25.7 (m 24.3 / 28.8)
//   [N,K] 2   169 x 128, K 15872 17.2 / 15.4  63 x 448, K 19680 17.4 / 19.9   64 x 64, K 191744 35 / 125
//         2, few columns   56 x 88, K 20992 23.5 / 16.7   127 x 64, K 23960 18.7 / 25.2
//         3   120 x 544, K 10304 16.4 / 13.8 (m 17.2 / 17.7)   53 x 1352, K 11232 16.6 / 16.7 (m 17.6 / 22.9)   209 x 376, K 12552 18.6 / 21.8 (m 20.7 / 24.6)
//         4   167 x 1224, K 8808 22.0 / 19.4 (m 23.4 / 23.5)   117 x 1336, K 9040 20.1 / 21.6 (m 24.4 / 26.9)   190 x 1112, K 21464 33 / 43
//         6   120 x 3792, K 4744 20.3 / 18.9 (m 24.5 / 24.5)   128 x 3096, K 5600 19.4 / 20.3 (m 23.4 / 26.3)
//         6, full   40 x 7640, K 6872 27.0 / 24.4 (m 34.7 / 29.9)   38 x 7928, K 10440 36.1 / 33.9 (m 53.9 / 49.9)   45 x 7600, K 11744 34.7 / 35.0 (m 47.9 / 52.4)
//         8   205 x 4088, K 4032 20.0 / 18.7 (m 23.0 / 21.2)   109 x 5160, K 4568 21.9 / 25.6 (m 27.9 / 33.4)   205 x 4008, K 9736 40 / 44; past the line 45
//             sizes 0.92 times
//   up to 32 rows against gemm_skinny.hpp ([N,K])   19 x 224, K 10048 9.5 / 8.9   15 x 320, K 13952 10.2 / 12.6
//   and against slices of 256 columns ([K,N])       26 x 512, K 6016 13.6 / 12.8   4 x 256, K 9600 14.2 / 18.0
static bool few_rows_slices_ahead(const GemmParams &p, const FewRowsTile &t) {
  const int64_t cost = t.rounds * (t.mt + t.nt);
  const bool full = p.M <= 64 && p.N >= 6784; // at a cost of 6: 64 x 32 tiles on nearly all compute units
  if (p.trans_b) {
    const int64_t k = cost <= 2 ? (p.N <= 128 ? 23040 : 16384) : cost == 3 ? 11776 : cost == 4 ? 8832 : cost <= 6 ? (full ? 11264 : 5120) : 3968;
    return p.K > (p.M <= 32 && k > 10240 ? 10240 : k);
  }
  const int64_t k = cost <= 2 ? (p.N <= 24 ? 24576 : p.N <= 40 ? 16384 : 5888) : cost == 3 ? 4608 : cost == 4 ? 4352 : cost == 5 ? 4096 : cost == 6 ? (full ? 5376 : 3840) : 3584;
  return p.K > (p.M < 32 && k < 6144 ? 6144 : k);
}

// Takes the call when the shape is this kernel's (returns -1 otherwise: the other kernels handle it).  slices: another kernel cuts
// this call's K over workgroups, and the workspace for it is there.
template <int ES> static int launch_few_rows(const GemmParams *pp, hipStream_t stream, bool dry, GemmTileConfig *cfg, bool slices) {
  GemmParams p = *pp;
  const int out_es = p.out_dt == DT_BF16 ? 2 : 4, res_es = p.residual_dt == DT_BF16 ? 2 : 4;
  auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  if (p.cfg_tile || p.cfg_split_k || p.cfg_waves) // a caller's MatmulConfig names another kernel's tile
    return -1;
  if (p.M < 1 || p.M > (ES == 1 ? 2048 : 256) || p.K < 1 || p.K % (16 / ES) != 0 || p.N % (ES == 2 && p.trans_b ? 4 : 16 / ES) != 0 || !al16(p.A) || !al16(p.B) ||
      !al16(p.C) || (p.lda * ES) % 16 != 0 || (p.ldb * ES) % 16 != 0 || (p.ldc * out_es) % 16 != 0 || (ES == 1 && (p.trans_b || p.residual)) ||
      (ES == 2 && p.out_dt == DT_S32) || (p.residual && p.residual_dt != DT_BF16 && p.residual_dt != DT_F32))
    return -1;
  const int64_t nbatch = p.batch > 1 ? p.batch : 1;
  if (nbatch > 65535 || p.N > (int64_t)1 << 28 || p.K > (int64_t)1 << 30)
    return -1;
  if (nbatch == 1)
    p.a_bs = p.b_bs = p.c_bs = 0;
  else if ((p.a_bs * ES) % 16 != 0 || (p.b_bs * ES) % 16 != 0 || (p.c_bs * out_es) % 16 != 0 || (p.residual && (p.c_bs * res_es) % 16 != 0))
    return -1;
  // a stage's rows reachable with 32-bit byte offsets
  if (p.lda * ES * 64 >= (int64_t)1 << 31 || p.ldb * ES * (p.trans_b ? 64 : 128) >= (int64_t)1 << 31)
    return -1;
  const FewRowsTile t = few_rows_tile(p.M, p.N, nbatch);
  if (t.blocks * nbatch > (int64_t)1 << 22) // (a grid has less than 2^32 threads)
    return -1;
  if (!few_rows_wanted<ES>(p, t) || (slices && few_rows_slices_ahead(p, t)))
    return -1;
  if (cfg) {
    GemmTileConfig c{};
    c.kernel = GK_FEW_ROWS, c.bm = 16 * t.mt, c.bn = 16 * t.nt, c.kbytes = 128, c.stages = t.stages;
    c.waves_m = c.waves_n = 1, c.wave_m = c.bm, c.wave_n = c.bn, c.mfma_m = c.mfma_n = 16, c.mfma_k = 64 / ES;
    c.split_k = 1, c.group_m = 1, c.workgroups = (int32_t)t.blocks;
    *cfg = c;
  }
  if (dry)
    return 0;
  const dim3 grid((unsigned)((t.blocks * nbatch + 7) / 8 * 8)), block(64 * t.waves);
#define GCMI_FEW_LAUNCH(TB, MT, NT, W, D)                                                                                \
  if (t.mt == MT && t.nt == NT)                                                                                           \
    hipLaunchKernelGGL((gemm_few_rows_kernel<ES, TB, MT, NT, W, D>), grid, block, 0, stream, p);
#define GCMI_FEW_ALL(TB)                                                                                              \
  GCMI_FEW_LAUNCH(TB, 1, 1, 8, 2) GCMI_FEW_LAUNCH(TB, 2, 1, 8, 2) GCMI_FEW_LAUNCH(TB, 4, 1, 4, 3)            \
  GCMI_FEW_LAUNCH(TB, 1, 2, 4, 3) GCMI_FEW_LAUNCH(TB, 2, 2, 4, 3) GCMI_FEW_LAUNCH(TB, 4, 2, 4, 3)            \
  GCMI_FEW_LAUNCH(TB, 1, 4, 4, 3) GCMI_FEW_LAUNCH(TB, 2, 4, 4, 3) GCMI_FEW_LAUNCH(TB, 4, 4, 4, 2)
  if (ES == 2 && p.trans_b) {
    if constexpr (ES == 2) {
      GCMI_FEW_ALL(true)
    }
  } else {
    GCMI_FEW_ALL(false)
  }
#undef GCMI_FEW_ALL
#undef GCMI_FEW_LAUNCH
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

} // namespace gcmi
