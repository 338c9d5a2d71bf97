// f32 GEMM on the f32 matrix instruction (f32 multiply-add throughout; no
// reduced precision) and the batch-reduce microkernel with the reference's
// operand layouts.
//
// gemm_f32_mfma_kernel, gemm_f32_small_kernel: C[M,N] = act(beta*C + A.B + bias),
// any sizes; either operand contiguous along k or along its own dimension, so
// that transpose_a / transpose_b of onednn_graph.matmul
// (lib/gc/Transforms/OneDNNGraphToLinalg.cpp:421-499) need no copy.
//
// brgemm_kernel: C[m*LDC+n] (+)= sum_i sum_k a(i,m,k) * b(i,k,n) with
//   f32 : b at i*stride_b + k*LDB + n
//   bf16: b at i*stride_b + (k - k%2)*LDB + 2n + k%2      (VNNI-2)
//   8bit: b at i*stride_b + (k - k%4)*LDB + 4n + k%4      (VNNI-4)
// (lib/gc/ExecutionEngine/CPURuntime/Microkernel/BrgemmNaive.cpp:46-140).
// Microkernel calls are small (typically 32x32x32 with a batch of 8-16); one
// thread per C element, operands staged through LDS, batch-major then k ascending as the reference sums, and
// every product and every sum rounded on its own (no fused multiply-add: the
// reference's loop is plain C++ built for baseline x86-64, which has none), so
// f32 results equal the reference's bit for bit; bf16 products are exact in f32
// and integer sums are exact anyway.
#include "common.hpp"
#include <math.h>
#include <type_traits>
#include "gemm_params.h"

#define GCMI_GLB __attribute__((address_space(1)))

namespace gcmi {

typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4))); // 16 bytes from any 4-byte aligned address

// One operand's side of a K slice: fetched to registers (float4 chunks, one slice ahead), stashed in LDS, read back as
// matrix operands.  KC: the operand is contiguous along k and lies in LDS as [row][k] -- one ds_read_b128 gives a lane
// the four k it contributes to a step (k = 4 * (lane / MT) + 0 .. 3: 8 or 16 deep for 32 x 32 or 16 x 16 products); else it is contiguous along its own
// dimension, lies in LDS as [k][column] and is read with four ds_read_b32.  Both sides use the same k in the same
// matrix instruction, which is all a sum needs, so neither layout is transposed on the way.
// Rows or chunks past the edge read the last valid ones instead (their products land in results nobody stores); a
// chunk cut by the edge reads the last four and moves them into place.
template <int BX, int BK, bool KC> struct F32Tile {
  // four floats of padding spread the rows over the banks (exchanging chunks within unpadded rows: 3 % slower)
  static constexpr int PITCH = KC ? BK + 4 : BX + 4, SIZE = KC ? BX * PITCH : BK * PITCH;
  static constexpr int PER = BX * BK / 4 / 256; // chunks per thread and slice
  static_assert(PER >= 1, "a slice is at least one chunk per thread");
  const float *src[PER]; // next slice's chunk
  int shift;             // !KC: places the chunk was moved back because the edge cuts it (the same for all chunks)
  bool cut;              // !KC: some chunk of this tile is cut (wave-uniform)
  int64_t step, ks;      // elements from slice to slice, from k to k
  f32x4_t r[2][PER];     // two slices in flight

  static __device__ __forceinline__ int x_of(int e) {
    const int idx = threadIdx.x + 256 * e;
    return KC ? idx / (BK / 4) : 4 * (idx % (BX / 4));
  }
  static __device__ __forceinline__ int k_of(int e) {
    const int idx = threadIdx.x + 256 * e;
    return KC ? 4 * (idx % (BK / 4)) : idx / (BX / 4);
  }
  __device__ __forceinline__ void init(const float *base, int64_t x0, int64_t X, int64_t xs, int64_t kstride) {
    ks = kstride, step = (int64_t)BK * kstride, shift = 0, cut = !KC && X - x0 < BX && X % 4 != 0;
    static_assert(KC || 256 % (BX / 4) == 0, "all chunks of a thread cover the same columns");
#pragma unroll
    for (int e = 0; e < PER; e++) {
      int64_t g = x0 + x_of(e);
      if constexpr (KC) {
        g = g < X ? g : X - 1;
      } else { // X >= 4
        const int64_t left = X - g;
        shift = left > 0 && left < 4 ? 4 - (int)left : 0;
        g = left >= 4 ? g : X - 4;
      }
      src[e] = base + g * xs + k_of(e) * kstride;
    }
  }
  __device__ __forceinline__ void fetch(int q) { // a whole slice, into register set q
#pragma unroll
    for (int e = 0; e < PER; e++) {
      r[q][e] = *reinterpret_cast<const f32x4u_t *>(src[e]);
      src[e] += step;
    }
  }
  __device__ __forceinline__ void fetch_tail(int q, int left) { // the last `left` < BK k, zero behind them
#pragma unroll
    for (int e = 0; e < PER; e++) {
#pragma unroll
      for (int c = 0; c < 4; c++)
        r[q][e][c] = k_of(e) + (KC ? c : 0) < left ? src[e][c] : 0.0f;
    }
  }
  __device__ __forceinline__ void stash(int q, float *lds) {
#pragma unroll
    for (int e = 0; e < PER; e++) {
      f32x4_t v = r[q][e];
      if constexpr (KC) {
        *reinterpret_cast<f32x4_t *>(&lds[x_of(e) * PITCH + k_of(e)]) = v;
      } else {
        if (cut) {
          const f32x4_t u = v;
          v[0] = shift == 0 ? u[0] : shift == 1 ? u[1] : shift == 2 ? u[2] : u[3];
          v[1] = shift == 0 ? u[1] : shift == 1 ? u[2] : u[3];
          v[2] = shift == 0 ? u[2] : u[3];
        }
        *reinterpret_cast<f32x4_t *>(&lds[k_of(e) * PITCH + x_of(e)]) = v;
      }
    }
  }
  // the four operand values of row/column x at k .. k + 3
  static __device__ __forceinline__ f32x4_t frag(const float *lds, int x, int k) {
    if constexpr (KC)
      return *reinterpret_cast<const f32x4_t *>(&lds[x * PITCH + k]);
    f32x4_t v;
#pragma unroll
    for (int c = 0; c < 4; c++)
      v[c] = lds[(k + c) * PITCH + x];
    return v;
  }
};

// One result: beta, bias, activation.
__device__ __forceinline__ void f32_store(const F32GemmParams &p, int64_t m, int64_t n, float x) {
  if (p.beta != 0.0f)
    x = x + p.C[m * p.ldc + n];
  if (p.bias)
    x = x + p.bias[n];
  p.C[m * p.ldc + n] = apply_act(x, p.act);
}

// BM x BN tile of a workgroup of 4 waves, WM x WN of them over the tile and WK over a slice of BK k (their partial sums
// are added through LDS at the end).  v_mfma_f32_32x32x2_f32: 256 flop per clock and compute unit (157 TFLOP/s), twice
// the vector ALU; a 64 x 64 tile needs 16 bytes per clock of operands, so nothing but the issue of these instructions
// should bound it.  MT: side of the matrix instruction's tile (16: the k of a step and their order are those of the
// small kernel below).  Two slices are in flight in registers behind the one in LDS (with one: 8 % slower, a load then has
// less time than memory takes), the barrier of a slice lies between its last products with the writes in front and the
// next slice's first reads behind it.  At 4096^3 the matrix pipes are 84 % busy: 1034 us = 133 TFLOP/s (1056 us on the
// same board when A was transposed on its way into LDS, one slice ahead).  1111 tokens through 1000 x 3000 x 1000 x 500:
// 177 us (470 on vector FMAs, which were all that sizes off the tile took).  v_mfma_f32_16x16x4_f32 in the large tiles: up to 10 % slower (more registers); in the 32 x 32 tile level.
template <int MT, int BM, int BN, int WM, int WN, int WK, int BK, bool AKC, bool BKC>
__global__ __launch_bounds__(256) void gemm_f32_mfma_kernel(F32GemmParams p) {
  constexpr int TM = BM / WM / MT, TN = BN / WN / MT, KW = BK / WK; // MT x MT tiles of a wave, its k of a slice
  constexpr int DEEP = 256 / MT, STEPS = KW / DEEP, R = MT * MT / 64; // k of a step, results per lane and tile
  static_assert(WM * WN * WK == 4 && KW % DEEP == 0, "4 waves, whole steps");
  typedef float acc_t __attribute__((ext_vector_type(R)));
  typedef F32Tile<BM, BK, AKC> TA;
  typedef F32Tile<BN, BK, BKC> TB;
  constexpr int STAGE = TA::SIZE + TB::SIZE;
  constexpr int RED = (WK - 1) * BM * BN;
  __shared__ __attribute__((aligned(16))) float smem[2 * STAGE > RED ? 2 * STAGE : RED];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wk = wave % WK, wn = (wave / WK) % WN, wm = wave / (WK * WN);
  const int lx = lane % MT, lk = lane / MT;
  // workgroup i runs on XCD i % 8: each XCD walks its own run of tiles, columns of 8 tile rows at a time
  const int64_t mt = (p.M + BM - 1) / BM, nt = (p.N + BN - 1) / BN, tiles = mt * nt;
  const int64_t t = (int64_t)(blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (t >= tiles)
    return;
  const int64_t group = t / (8 * nt), rows = mt - 8 * group < 8 ? mt - 8 * group : 8, in = t - group * 8 * nt;
  const int64_t m0 = (8 * group + in % rows) * BM, n0 = in / rows * BN;
  p.A += (int64_t)blockIdx.z * p.a_bs, p.B += (int64_t)blockIdx.z * p.b_bs, p.C += (int64_t)blockIdx.z * p.c_bs;
  TA ta;
  TB tb;
  ta.init(p.A, m0, p.M, p.a_rs, p.a_cs);
  tb.init(p.B, n0, p.N, p.b_cs, p.b_rs);
  acc_t acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; i++)
#pragma unroll
    for (int j = 0; j < TN; j++)
#pragma unroll
      for (int r = 0; r < R; r++)
        acc[i][j][r] = 0.0f;
  const int xa = wm * TM * MT + lx, xb = wn * TN * MT + lx;
  f32x4_t a[2][TM], b[2][TN]; // operands of this step and the next
  auto load = [&](int q, int step) { // of the slice in slot q
    const float *as = smem + q * STAGE, *bs = as + TA::SIZE;
    const int s = (q * STEPS + step) & 1, k = wk * KW + DEEP * step + 4 * lk;
#pragma unroll
    for (int i = 0; i < TM; i++)
      a[s][i] = TA::frag(as, xa + i * MT, k);
#pragma unroll
    for (int j = 0; j < TN; j++)
      b[s][j] = TB::frag(bs, xb + j * MT, k);
  };
  auto products = [&](int s, int c) {
#pragma unroll
    for (int i = 0; i < TM; i++)
#pragma unroll
      for (int j = 0; j < TN; j++)
        if constexpr (MT == 32)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[s][i][c], b[s][j][c], acc[i][j], 0, 0, 0);
        else
          acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[s][i][c], b[s][j][c], acc[i][j], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0); // reads and writes keep their places between the products
  };
  // slice s lies in slot s % 2 (offset 0 or STAGE); slice s + 1 is in register set (s + 1) % 2 or on its way there,
  // slice s + 2 is requested into set s % 2 at the start: two slices' worth of products to hide a load behind
  const int64_t whole = p.K / BK;
  const int tail = (int)(p.K - whole * BK);
  const int64_t slices = whole + (tail ? 1 : 0);
  auto fetch = [&](int q, int64_t s) {
    if (s < whole)
      ta.fetch(q), tb.fetch(q);
    else if (s < slices)
      ta.fetch_tail(q, tail), tb.fetch_tail(q, tail);
  };
  auto stash = [&](int q) {
    ta.stash(q, smem + q * STAGE);
    tb.stash(q, smem + q * STAGE + TA::SIZE);
  };
  auto slice = [&](int q, bool next) {
#pragma unroll
    for (int step = 0; step < STEPS - 1; step++) {
      load(q, step + 1);
#pragma unroll
      for (int c = 0; c < 4; c++)
        products((q * STEPS + step) & 1, c);
    }
    const int last = (q * STEPS + STEPS - 1) & 1;
    products(last, 0);
    if (next)
      stash(q ^ 1);
    products(last, 1);
    if (next) {
      __syncthreads();
      load(q ^ 1, 0); // the next slice's first operands, under the last products of this one
    }
    products(last, 2);
    products(last, 3);
  };
  if (slices > 0) {
    fetch(0, 0);
    fetch(1, 1);
    stash(0);
    __syncthreads();
    load(0, 0);
    int64_t s = 0;
    for (; s + 3 < whole; s += 2) {
#pragma unroll
      for (int q = 0; q < 2; q++) {
        ta.fetch(q), tb.fetch(q);
        __builtin_amdgcn_sched_barrier(0);
        slice(q, true);
      }
    }
    for (; s < slices; s += 2) {
#pragma unroll
      for (int q = 0; q < 2; q++)
        if (s + q < slices) {
          fetch(q, s + q + 2);
          slice(q, s + q + 1 < slices);
        }
    }
  }
  if constexpr (WK > 1)
    __syncthreads(); // the operand slots become the reduction's
  if constexpr (WK > 1) { // the waves' shares of K, added in ascending order of wk
    float *mine = smem + (wm * WN + wn) * (WK - 1) * TM * TN * R * 64 + lane;
    if (wk > 0) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int r = 0; r < R; r++)
            mine[(((wk - 1) * TM + i) * TN + j) * R * 64 + r * 64] = acc[i][j][r];
    }
    __syncthreads();
    if (wk > 0)
      return;
#pragma unroll
    for (int w = 0; w < WK - 1; w++)
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int j = 0; j < TN; j++)
#pragma unroll
          for (int r = 0; r < R; r++)
            acc[i][j][r] += mine[((w * TM + i) * TN + j) * R * 64 + r * 64];
  }
  // lane (lx, lk) holds column lx and rows 8 * (r / 4) + 4 * lk + r % 4 of every tile
#pragma unroll
  for (int j = 0; j < TN; j++) {
    const int64_t n = n0 + (wn * TN + j) * MT + lx;
    if (n < p.N) {
#pragma unroll
      for (int i = 0; i < TM; i++)
#pragma unroll
        for (int r = 0; r < R; r++) {
          const int64_t m = m0 + (wm * TM + i) * MT + 8 * (r >> 2) + 4 * lk + (r & 3);
          if (m < p.M)
            f32_store(p, m, n, acc[i][j][r]);
        }
    }
  }
}

// Small problems: what counts is the chain launch -> loads -> sums -> store.  A workgroup owns one 16 x 16 tile, its
// four waves take every fourth 16-deep step of K straight from memory into v_mfma_f32_16x16x4_f32 operands (lane l:
// row/column l % 16, and k = 4 * (l / 16) .. + 3 of the step as four operand values), up to eight steps in flight per wave,
// no LDS and no barrier until the four partial sums are added.  Kernel alone, us: 128 x 256, K 512 (128 workgroups) 4.15, 532 x
// 492, K 1068 17.0, 154 x 737, K 1872 16.0, 1000 x 64, K 3000 12.6 (4.31, 20.0, 18.1 and 15.1 when a wave waited for eight steps
// at a time and then took the rest of K step by step; 4.50, 20.7, 16.6 and 13.3 when all but its first step's loads were flat
// ones, each wait for all of them); sixteen steps in flight are the slower choice where workgroups share a compute unit.
static constexpr int64_t F32_SMALL_GRID = 1 << 23; // workgroups of a grid's first dimension, at most: 2^32 threads are too many
// WIDE: a lane's place in a step may lie more than 2^31 bytes behind the step's first element; else it is a 32-bit offset on
// a scalar address (with 64-bit addresses in the lanes every load in flight takes two registers more).
template <bool AKC, bool BKC, bool WIDE> __global__ __launch_bounds__(256) void gemm_f32_small_kernel(F32GemmParams p) {
  constexpr int U = 4;
  __shared__ float red[3][256];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), l16 = lane & 15, lq = lane >> 4;
  // The size of the grid is a constant, and workgroups past the last tile (a grid of more than one row) compute rows that
  // nobody stores: reading the size, or leaving early, puts a second wait for kernel arguments in front of the loads of
  // every workgroup (0.2 us a launch).
  const int64_t nt = (p.N + 15) / 16, t = blockIdx.x + (int64_t)blockIdx.y * F32_SMALL_GRID;
  const int64_t m0 = t / nt * 16, n0 = t % nt * 16;
  p.C += (int64_t)blockIdx.z * p.c_bs;
  // rows past the last one read the last one (a tile past the last one: its own rows' clamp)
  const int64_t ma = m0 < p.M ? m0 : p.M - 1;
  const int ra = ma + l16 < p.M ? l16 : (int)(p.M - 1 - ma), rb = n0 + l16 < p.N ? l16 : (int)(p.N - 1 - n0);
  // (global by their type: behind the pins below the compiler cannot tell, and waits for all flat loads together)
  typedef typename std::conditional<WIDE, int64_t, uint32_t>::type off_t;
  typedef GCMI_GLB const char *mem_t;
  mem_t a = (mem_t)(p.A + (int64_t)blockIdx.z * p.a_bs + ma * p.a_rs), b = (mem_t)(p.B + (int64_t)blockIdx.z * p.b_bs + n0 * p.b_cs);
  off_t la[AKC ? 1 : 4], lb[BKC ? 1 : 4]; // the lane's four k, or its four contiguous ones
#pragma unroll
  for (int c = 0; c < (AKC ? 1 : 4); c++)
    la[c] = 4 * ((off_t)ra * (off_t)p.a_rs + (off_t)(4 * lq + c) * (off_t)(AKC ? 1 : p.a_cs));
#pragma unroll
  for (int c = 0; c < (BKC ? 1 : 4); c++)
    lb[c] = 4 * ((off_t)rb * (off_t)p.b_cs + (off_t)(4 * lq + c) * (off_t)(BKC ? 1 : p.b_rs));
  f32x4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
  auto load = [](mem_t s, const auto &o) -> f32x4_t {
    if constexpr (sizeof(o) == sizeof(off_t))
      return *(GCMI_GLB const f32x4u_t *)(s + o[0]);
    else
      return f32x4_t{*(GCMI_GLB const float *)(s + o[0]), *(GCMI_GLB const float *)(s + o[1]), *(GCMI_GLB const float *)(s + o[2]),
                     *(GCMI_GLB const float *)(s + o[3])};
  };
  auto load_end = [](mem_t s, const auto &o, int left) -> f32x4_t {
    f32x4_t v;
#pragma unroll
    for (int c = 0; c < 4; c++) {
      constexpr bool contig = sizeof(o) == sizeof(off_t);
      v[c] = 0.0f;
      if (c < left)
        v[c] = *(GCMI_GLB const float *)(contig ? s + o[0] + 4 * c : s + o[contig ? 0 : c]);
    }
    return v;
  };
  // This wave's whole steps are wave, wave + 4, ...; the step that K ends inside of, if it does, is behind some wave's last.
  // Four steps are multiplied (a chain of 16 sums) while the next four are on their way, and what is left of K is one more
  // round of loads.
  const int steps = (int)((p.K / 16 - wave + 3) >> 2), left = (int)(p.K & 15);
  const bool ends = left != 0 && (int)((p.K >> 4) & 3) == wave;
  const int64_t a_step = 256 * (AKC ? 1 : p.a_cs), b_step = 256 * (BKC ? 1 : p.b_rs);
  a += 64 * wave * (AKC ? 1 : p.a_cs), b += 64 * wave * (BKC ? 1 : p.b_rs);
  f32x4_t va[2][U], vb[2][U], ea, eb;
  // (the addresses are scalars that go from step to step, the lane's offsets 32 bits beside them: worked out or widened ahead,
  // as the compiler would, they fill the registers)
  auto step = [&](f32x4_t &x, f32x4_t &y) {
    x = load(a, la), y = load(b, lb);
    a += a_step, b += b_step;
    asm volatile("" : "+s"(a), "+s"(b));
  };
  auto fetch = [&](int q) { // U steps
    if constexpr (!WIDE) {
#pragma unroll
      for (auto &o : la)
        asm volatile("" : "+v"(o));
#pragma unroll
      for (auto &o : lb)
        asm volatile("" : "+v"(o));
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      step(va[q][u], vb[q][u]);
    __builtin_amdgcn_sched_barrier(0); // all loads first
  };
  auto product = [&](const f32x4_t &x, const f32x4_t &y) {
#pragma unroll
    for (int c = 0; c < 4; c++)
      acc = __builtin_amdgcn_mfma_f32_16x16x4f32(x[c], y[c], acc, 0, 0, 0);
  };
  auto products = [&](int q) {
#pragma unroll
    for (int u = 0; u < U; u++)
      product(va[q][u], vb[q][u]);
    __builtin_amdgcn_sched_barrier(0);
  };
  auto fetch_rest = [&](int q, int n) { // n steps, fewer than U, and the end of K
#pragma unroll
    for (int u = 0; u < U - 1; u++)
      if (u < n)
        step(va[q][u], vb[q][u]);
    if (ends) {
      ea = load_end(a, la, left - 4 * lq);
      eb = load_end(b, lb, left - 4 * lq);
    }
  };
  auto products_rest = [&](int q, int n) {
#pragma unroll
    for (int u = 0; u < U - 1; u++)
      if (u < n)
        product(va[q][u], vb[q][u]);
    if (ends)
      product(ea, eb);
  };
  if (steps < U) {
    fetch_rest(0, steps);
    products_rest(0, steps);
  } else {
    int n = steps - U; // steps not asked for yet
    fetch(0);
    for (; n >= 2 * U; n -= 2 * U) {
      fetch(1);
      products(0);
      fetch(0);
      products(1);
    }
    if (n >= U) {
      fetch(1);
      products(0);
      fetch_rest(0, n - U);
      products(1);
      products_rest(0, n - U);
    } else {
      fetch_rest(1, n);
      products(0);
      products_rest(1, n);
    }
  }
  if (wave > 0)
#pragma unroll
    for (int r = 0; r < 4; r++)
      red[wave - 1][r * 64 + lane] = acc[r];
  __syncthreads();
  if (wave > 0)
    return;
#pragma unroll
  for (int r = 0; r < 4; r++) {
    float x = acc[r];
#pragma unroll
    for (int w = 0; w < 3; w++)
      x += red[w][r * 64 + lane];
    const int64_t m = m0 + 4 * lq + r, n = n0 + l16; // lane l holds column l % 16 and rows 4 * (l / 16) + r
    if (m < p.M && n < p.N)
      f32_store(p, m, n, x);
  }
}

// A short K (see f32_plan): products on the vector ALU.  BT x BT workgroup tile (BT = 64, 32 or 16: small problems
// take small tiles so that more compute units take part), 256 threads, (BT/16)^2 outputs per thread, 32-deep K slices
// through LDS: with one slice a workgroup is one load, one barrier and one store, where the matrix kernels' slices of 32
// and 64 k come half empty.
template <int BT> __global__ __launch_bounds__(256) void gemm_f32_fma_kernel(F32GemmParams p) {
  constexpr int BK = 32, MT = BT / 16, PER = BT * BK / 256; // elements per thread per operand slice
  __shared__ float As[BK][BT + 4];
  __shared__ float Bs[BK][BT + 4];
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int64_t m0 = (int64_t)blockIdx.y * BT, n0 = (int64_t)blockIdx.x * BT;
  p.A += (int64_t)blockIdx.z * p.a_bs, p.B += (int64_t)blockIdx.z * p.b_bs, p.C += (int64_t)blockIdx.z * p.c_bs;
  // slice element e of this thread: (row/col within the tile, k within the slice);
  // the contiguous direction of each operand runs along consecutive threads
  int am[PER], ak[PER], bn[PER], bk[PER];
#pragma unroll
  for (int e = 0; e < PER; e++) {
    const int idx = threadIdx.x + 256 * e;
    if (p.a_cs == 1) {
      ak[e] = idx % BK;
      am[e] = idx / BK;
    } else {
      am[e] = idx % BT;
      ak[e] = idx / BT;
    }
    if (p.b_rs == 1 && p.b_cs != 1) {
      bk[e] = idx % BK;
      bn[e] = idx / BK;
    } else {
      bn[e] = idx % BT;
      bk[e] = idx / BT;
    }
  }
  float ra[PER], rb[PER];
  auto fetch = [&](int64_t k0) {
#pragma unroll
    for (int e = 0; e < PER; e++) {
      const int64_t gm = m0 + am[e], gk = k0 + ak[e];
      ra[e] = (gm < p.M && gk < p.K) ? p.A[gm * p.a_rs + gk * p.a_cs] : 0.0f;
      const int64_t gn = n0 + bn[e], gk2 = k0 + bk[e];
      rb[e] = (gn < p.N && gk2 < p.K) ? p.B[gk2 * p.b_rs + gn * p.b_cs] : 0.0f;
    }
  };
  float acc[MT][MT] = {};
  fetch(0);
  for (int64_t k0 = 0; k0 < p.K; k0 += BK) {
#pragma unroll
    for (int e = 0; e < PER; e++) {
      As[ak[e]][am[e]] = ra[e];
      Bs[bk[e]][bn[e]] = rb[e];
    }
    __syncthreads();
    if (k0 + BK < p.K)
      fetch(k0 + BK);
#pragma unroll
    for (int k = 0; k < BK; k++) { // k ascending per output element
      float a[MT], b[MT];
#pragma unroll
      for (int i = 0; i < MT; i++)
        a[i] = As[k][ty * MT + i];
#pragma unroll
      for (int j = 0; j < MT; j++)
        b[j] = Bs[k][tx * MT + j];
#pragma unroll
      for (int i = 0; i < MT; i++)
#pragma unroll
        for (int j = 0; j < MT; j++)
          acc[i][j] = fmaf(a[i], b[j], acc[i][j]);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < MT; i++) {
    int64_t m = m0 + ty * MT + i;
    if (m >= p.M)
      continue;
#pragma unroll
    for (int j = 0; j < MT; j++) {
      int64_t n = n0 + tx * MT + j;
      if (n >= p.N)
        continue;
      float x = acc[i][j];
      if (p.beta != 0.0f)
        x = x + p.C[m * p.ldc + n];
      if (p.bias)
        x = x + p.bias[n];
      p.C[m * p.ldc + n] = apply_act(x, p.act);
    }
  }
}

struct BrgemmParams {
  const void *A, *B;
  void *C;
  int64_t M, N, K, LDA, LDB, LDC, stride_a, stride_b;
  int32_t num, beta_zero, dtA, dtB;
};

// One workgroup = one 16 x 16 tile of C, one thread per element.  The terms of an element's sum keep the reference's
// order (batch-major, k ascending, each product and each sum rounded on its own), so the only freedom is where the
// operands come from: the workgroup stages BRG_CH terms' worth of its 16 rows of A and 16 columns of B in LDS as
// widened values (f32, or s32 for the 8-bit types), both with the terms contiguous so that four terms come out of
// one 16-byte read per operand -- and the loads of the next chunk are in flight in registers while this chunk is
// summed.  A chunk is a run of whole batches when K is small (the usual 32 x 32 x 32 call) or a slice of one batch's
// K.  K tails of the packed layouts are never read and never added (adding a zero would turn a -0 sum into +0).
// A wave issues a vector instruction that needs its predecessor's result only every 8-9 cycles, so the chain of num*K dependent sums
// is the floor; everything else is kept short: element offsets are worked out once, a chunk adds two scalars.
static constexpr int BRG_CH = 128, BRG_PITCH = BRG_CH + 4, BRG_PER = 16 * BRG_CH / 256;

template <typename ACC, int V> // V: the k elements packed beside each other in B (1 f32, 2 bf16, 4 8-bit)
__global__ __launch_bounds__(256) void brgemm_kernel(BrgemmParams p) {
#pragma clang fp contract(off) // a product and the sum it goes into are rounded separately, as the reference's are
  __shared__ __attribute__((aligned(16))) ACC As[16][BRG_PITCH]; // [row of the tile][term of the chunk]
  __shared__ __attribute__((aligned(16))) ACC Bs[16][BRG_PITCH]; // [column of the tile][term of the chunk]
  const int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * 16, m0 = (int64_t)blockIdx.y * 16;
  // chunk geometry: kc terms of K per batch and chunk, nb batches per chunk; chunks run batch group by batch group
  // and, inside one, K slice by K slice
  const int kc = p.K < BRG_CH ? (int)p.K : BRG_CH;
  const int nb = p.K < BRG_CH ? BRG_CH / (kc > 0 ? kc : 1) : 1;
  const int64_t kchunks = p.K > 0 ? (p.K + kc - 1) / kc : 0;
  const int64_t nchunks = ((p.num + nb - 1) / nb) * kchunks;
  const bool a_signed = p.dtA == DT_S8, b_signed = p.dtB == DT_S8;

  // Loads keep the raw element (a register each); widening waits until the value goes to LDS, one chunk later, so
  // that nothing between a load and the sums of the current chunk needs the loaded value.
  typedef typename std::conditional<V == 1, float, uint32_t>::type RAW;
  auto load = [&](const void *base, int64_t idx) -> RAW {
    if constexpr (V == 1)
      return ((const float *)base)[idx];
    else if constexpr (V == 2)
      return ((const uint16_t *)base)[idx];
    else
      return ((const uint8_t *)base)[idx];
  };
  auto widen = [&](RAW v, bool is_signed) -> ACC {
    if constexpr (V == 1)
      return v;
    else if constexpr (V == 2)
      return __uint_as_float(v << 16);
    else
      return is_signed ? (int)(v ^ 0x80u) - 0x80 : (int)v;
  };
  // Slot e of a chunk.  A: (row, term), terms along consecutive threads.  B: (term group, column, k within the
  // group), the order B lies in memory.  Term t of a chunk = (batch t / kc, k t % kc) relative to the chunk's first
  // batch and first k (a multiple of V, so the packed position of k does not depend on the chunk).
  int64_t a_off[BRG_PER], b_off[BRG_PER];
  int a_bat[BRG_PER], a_k[BRG_PER], b_bat[BRG_PER], b_k[BRG_PER];
#pragma unroll
  for (int e = 0; e < BRG_PER; e++) {
    const int idx = threadIdx.x + 256 * e;
    const int ta = idx % BRG_CH, tb = (idx / (16 * V)) * V + idx % V;
    const int kd = kc > 0 ? kc : 1;
    const int64_t m = m0 + idx / BRG_CH, n = n0 + (idx % (16 * V)) / V;
    a_bat[e] = (ta < nb * kc && m < p.M) ? ta / kd : 1 << 30, a_k[e] = ta % kd; // 1 << 30: never a valid batch
    b_bat[e] = (tb < nb * kc && n < p.N) ? tb / kd : 1 << 30, b_k[e] = tb % kd;
    a_off[e] = (int64_t)(ta / kd) * p.stride_a + m * p.LDA + a_k[e];
    b_off[e] = (int64_t)(tb / kd) * p.stride_b + (int64_t)(b_k[e] - b_k[e] % V) * p.LDB + V * n + b_k[e] % V;
  }
  RAW ra[BRG_PER], rb[BRG_PER];
  auto fetch = [&](int64_t b0, int64_t k0) {
    const int64_t a_chunk = b0 * p.stride_a + k0, b_chunk = b0 * p.stride_b + k0 * p.LDB;
    const int64_t bats = p.num - b0, ks = p.K - k0; // batches and k left from here
#pragma unroll
    for (int e = 0; e < BRG_PER; e++) {
      ra[e] = (a_bat[e] < bats && a_k[e] < ks) ? load(p.A, a_off[e] + a_chunk) : RAW(0);
      rb[e] = (b_bat[e] < bats && b_k[e] < ks) ? load(p.B, b_off[e] + b_chunk) : RAW(0);
    }
  };
  auto stash = [&]() {
#pragma unroll
    for (int e = 0; e < BRG_PER; e++) {
      const int idx = threadIdx.x + 256 * e;
      As[idx / BRG_CH][idx % BRG_CH] = widen(ra[e], a_signed);
      Bs[(idx % (16 * V)) / V][(idx / (16 * V)) * V + idx % V] = widen(rb[e], b_signed);
    }
  };
  auto term = [](ACC s, ACC a, ACC b) -> ACC {
    if constexpr (V == 4)
      return __mul24(a, b) + s; // 8-bit values: one 24-bit multiply-add, exact
    else
      return s + a * b;
  };
  const int64_t m = m0 + ty, n = n0 + tx;
  const bool mine = m < p.M && n < p.N;
  ACC *c = (ACC *)p.C + m * p.LDC + n;
  ACC s = (p.beta_zero || !mine) ? ACC(0) : *c;
  int64_t b0 = 0, k0 = 0, b0n = 0, k0n = 0; // this chunk's first batch and k, and the next chunk's
  auto advance = [&]() {
    k0n += kc;
    if (k0n >= p.K)
      k0n = 0, b0n += nb;
  };
  if (nchunks > 0) {
    fetch(0, 0);
    advance();
  }
  typedef ACC acc4 __attribute__((ext_vector_type(4)));
  for (int64_t ch = 0; ch < nchunks; ch++) {
    stash();
    __syncthreads();
    if (ch + 1 < nchunks)
      fetch(b0n, k0n);
    const int nbat = (int)((p.num - b0) < nb ? (p.num - b0) : nb);
    const int klen = (int)((p.K - k0) < kc ? (p.K - k0) : kc);
    for (int bi = 0; bi < nbat; bi++) {
      const int t0 = bi * kc;
      int k = 0;
      if ((kc & 3) == 0) { // every batch of the chunk starts on a 16-byte boundary
#pragma unroll 2
        for (; k + 4 <= klen; k += 4) {
          const acc4 a = *reinterpret_cast<const acc4 *>(&As[ty][t0 + k]);
          const acc4 b = *reinterpret_cast<const acc4 *>(&Bs[tx][t0 + k]);
          s = term(s, a.x, b.x);
          s = term(s, a.y, b.y);
          s = term(s, a.z, b.z);
          s = term(s, a.w, b.w);
        }
      }
      for (; k < klen; k++)
        s = term(s, As[ty][t0 + k], Bs[tx][t0 + k]);
    }
    __syncthreads();
    b0 = b0n, k0 = k0n;
    advance();
  }
  if (mine)
    *c = s;
}

} // namespace gcmi

using namespace gcmi;

// the kernel of one tile for the four operand layouts (A along k: + 2, B along k: + 1)
#define F32_LAYOUTS(...)                                                                                              \
  {gemm_f32_mfma_kernel<__VA_ARGS__, false, false>, gemm_f32_mfma_kernel<__VA_ARGS__, false, true>,                   \
   gemm_f32_mfma_kernel<__VA_ARGS__, true, false>, gemm_f32_mfma_kernel<__VA_ARGS__, true, true>}

static bool f32_a_along_k(const F32GemmParams &p) { return p.a_cs == 1; }
static bool f32_b_along_k(const F32GemmParams &p) { return p.b_rs == 1 && p.b_cs != 1; }
struct F32Plan {
  int tile;
  bool vector; // gemm_f32_fma_kernel
};
// The tile by estimated time (us, fitted to graph-replayed launches of 1 .. 2048 rows, 16 .. 3000 columns and K 16 .. 3000 on
// one MI355X; n tiles per compute unit, k = K / 1000; two constants where a lone workgroup of a compute unit is slower
// than one of several): tiles are dealt out evenly, a compute unit is done when the one with the most is, and a tile
// costs its start and its stores whatever K is.  1111 x 1000, K 3000, in us: 128 x 128 198, 64 x 64 100, 32 x 32 77;
// 4096^3: 1034, 1051, 1218; 1000 x 1000 x 1000: 75, 24-26, 29; 300 x 300, K 1000: 73, 23, 11.4 and 8.3 with 16 x 16 tiles;
// 1071 x 2048, K 16: 13, 8.7, 17, 17 (an estimate without the cost of a tile took 16 x 16 here).
// The two small tiles add an element's products in the same order, and so do the two large ones, and the vector
// kernel whatever its tile: which of the three is taken depends on one matrix, so a batch has the bits of its matrices
// multiplied one by one.
static F32Plan f32_plan(const F32GemmParams &p) {
  const double cus = gcmi_num_cus(), k = (double)p.K * 1e-3, nbatch = (double)(p.batch > 1 ? p.batch : 1);
  auto tiles = [&](int64_t t) { return (double)(((p.M + t - 1) / t) * ((p.N + t - 1) / t)); };
  auto us = [&](int tile, double batches) {
    const double n = batches * tiles(tile) / cus; // per compute unit
    switch (tile) {
    case 16: return 2.7 + fmax(3.8 * k, (0.38 + 2.7 * k) * n);
    case 32: return 4.6 + (1.3 + 4.6 * k) * ceil(n);
    case 64: return 4.5 + 1.1 * ceil(n) + k * fmax(18.3, 16.2 * ceil(n));
    default: return 7.5 + 4.0 * ceil(n) + k * fmax(63.0, 60.0 * ceil(n));
    }
  };
  // A K of one 32-deep slice and less than a round of 64 x 64 tiles: the vector kernel.  256 x 2048, K 32: 4.5 us, 5.6
  // on the best matrix tile; 512 x 2048: 8.5 and 5.9; K 40: 5.9 and 6.6, but 256 x 3000 7.2 and 6.8, 512 x 1500 7.4 and 6.8.
  if (p.K <= 32 && tiles(64) < cus && (p.M + 15) / 16 <= 65535)
    return {tiles(64) * nbatch >= cus ? 64 : tiles(32) * nbatch >= cus ? 32 : 16, true};
  // 16 bytes along m (A stored [K,M]) or n (B stored [K,N]) are a chunk of the tiles from 32 x 32 on: one must exist
  const bool chunk = (f32_a_along_k(p) || p.M >= 4) && (f32_b_along_k(p) || p.N >= 4);
  if (chunk && fmin(us(64, 1), us(128, 1)) < fmin(us(16, 1), us(32, 1)))
    return {us(128, nbatch) < us(64, nbatch) ? 128 : 64, false};
  return {chunk && us(32, nbatch) < us(16, nbatch) ? 32 : 16, false};
}

// what the launch below would choose (nothing is launched)
extern "C" int gcmi_launch_gemm_f32_config(const F32GemmParams *p, GemmTileConfig *cfg) {
  const F32Plan plan = f32_plan(*p);
  GemmTileConfig c{};
  c.kernel = GK_F32, c.bm = c.bn = plan.tile, c.split_k = 1, c.group_m = 8;
  c.workgroups = (int32_t)(((p->M + plan.tile - 1) / plan.tile) * ((p->N + plan.tile - 1) / plan.tile));
  c.stages = plan.vector || plan.tile == 16 ? 1 : 2;
  c.kbytes = plan.vector ? 128 : plan.tile == 16 ? 0 : plan.tile == 32 ? 256 : plan.tile == 64 ? 128 : 64;
  c.waves_m = c.waves_n = plan.tile >= 64 && !plan.vector ? 2 : 1;
  c.wave_m = c.wave_n = plan.tile / c.waves_m;
  if (!plan.vector)
    c.mfma_m = c.mfma_n = plan.tile >= 64 ? 32 : 16, c.mfma_k = plan.tile >= 64 ? 2 : 4;
  *cfg = c;
  return 0;
}

extern "C" int gcmi_launch_gemm_f32(const F32GemmParams *pp, hipStream_t stream) {
  F32GemmParams p = *pp;
  if (p.M <= 0 || p.N <= 0)
    return 0;
  const int64_t nbatch = p.batch > 1 ? p.batch : 1;
  if (nbatch > 65535)
    return 2;
  const F32Plan plan = f32_plan(p);
  int tile = plan.tile;
  const int layout = (f32_a_along_k(p) ? 2 : 0) + (f32_b_along_k(p) ? 1 : 0);
  if (plan.vector) {
    const dim3 grid((unsigned)((p.N + tile - 1) / tile), (unsigned)((p.M + tile - 1) / tile), (unsigned)nbatch);
    hipLaunchKernelGGL(tile == 64 ? gemm_f32_fma_kernel<64> : tile == 32 ? gemm_f32_fma_kernel<32> : gemm_f32_fma_kernel<16>, grid,
                       dim3(256), 0, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : 5;
  }
  if (tile == 16) {
    const int64_t all = ((p.N + 15) / 16) * ((p.M + 15) / 16), gx = all < F32_SMALL_GRID ? all : F32_SMALL_GRID;
    if ((all + gx - 1) / gx > 65535)
      return 2;
    const dim3 grid((unsigned)gx, (unsigned)((all + gx - 1) / gx), (unsigned)nbatch);
    // the last byte that a lane reads of a step, counted from the step's first
    auto far = [](int64_t xs, int64_t ks) { return 4 * (15 * xs + 15 * ks + 1) >= (int64_t)1 << 31; };
    const bool wide = far(p.a_rs, p.a_cs) || far(p.b_cs, p.b_rs);
    void (*const kernel[8])(F32GemmParams) = {gemm_f32_small_kernel<false, false, false>, gemm_f32_small_kernel<false, true, false>,
                                              gemm_f32_small_kernel<true, false, false>, gemm_f32_small_kernel<true, true, false>,
                                              gemm_f32_small_kernel<false, false, true>, gemm_f32_small_kernel<false, true, true>,
                                              gemm_f32_small_kernel<true, false, true>, gemm_f32_small_kernel<true, true, true>};
    hipLaunchKernelGGL(kernel[layout + (wide ? 4 : 0)], grid, dim3(256), 0, stream, p);
    return hipGetLastError() == hipSuccess ? 0 : 5;
  }
  static void (*const kernels[3][4])(F32GemmParams) = {F32_LAYOUTS(16, 32, 32, 1, 1, 4, 64),
                                                       F32_LAYOUTS(32, 64, 64, 2, 2, 1, 32),
                                                       F32_LAYOUTS(32, 128, 128, 2, 2, 1, 16)};
  auto per_xcd_of = [&](int t) { return (((p.M + t - 1) / t) * ((p.N + t - 1) / t) + 7) / 8; };
  while (tile < 128 && per_xcd_of(tile) * 8 >= 1 << 24) // too many for a grid dimension: a question of one matrix as well
    tile *= 2;
  const int64_t per_xcd = per_xcd_of(tile);
  if (per_xcd * 8 >= 1 << 24)
    return 2;
  hipLaunchKernelGGL(kernels[tile == 32 ? 0 : tile == 64 ? 1 : 2][layout], dim3((unsigned)(per_xcd * 8), 1, (unsigned)nbatch), dim3(256), 0, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

extern "C" int gcmi_launch_brgemm(const void *A, const void *B, void *C, int64_t M, int64_t N, int64_t K, int64_t LDA,
                                  int64_t LDB, int64_t LDC, int64_t stride_a, int64_t stride_b, int num, int beta_zero,
                                  int dtA, int dtB, hipStream_t stream) {
  if (M <= 0 || N <= 0)
    return 0;
  BrgemmParams p{A, B, C, M, N, K, LDA, LDB, LDC, stride_a, stride_b, num, beta_zero, dtA, dtB};
  dim3 grid((unsigned)((N + 15) / 16), (unsigned)((M + 15) / 16)), block(256);
  if (grid.y > 65535)
    return 2;
  if (dtA == DT_F32)
    hipLaunchKernelGGL((brgemm_kernel<float, 1>), grid, block, 0, stream, p);
  else if (dtA == DT_BF16)
    hipLaunchKernelGGL((brgemm_kernel<float, 2>), grid, block, 0, stream, p);
  else
    hipLaunchKernelGGL((brgemm_kernel<int32_t, 4>), grid, block, 0, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : 5;
}
