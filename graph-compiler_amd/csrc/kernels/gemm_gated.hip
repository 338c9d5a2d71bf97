// silu(A . gate^T) * (A . up^T) in one launch: the two products of a gated feed-forward layer with the ops between them
// (bf16, both weights stored [N,K], one shape and row length; the rounding points of the graph's separate ops).  As three
// launches the products are written and read back, each launch fills and drains the GPU by itself, and for few rows both
// products put their weights on two thirds of the compute units.
//   gemm_gated_rows_kernel  up to 64 rows (128 with narrow weights): streams the weights
//   gemm_gated_kernel       more: the 4-wave tiles with the hand-placed loop, half their columns for each product
#include "gemm_tile256.hpp"

namespace gcmi {

static constexpr int GR_KB = 256; // bytes of K per row and stage

// Up to 32, 64 or 128 rows (MT = 2, 4, 8).  The time is that of pulling the weights, which wants every compute unit to pull its
// share: a workgroup takes `cols` columns of both products, cols such that one round of workgroups holds them all (11008
// columns: 251 workgroups of 44, where 64-column panels of one product are 172).  8 waves; a stage is 128 elements of K: A and
// 2 x cols rows of weights, whole 256-byte rows, go to an LDS ring of up to four stages (16 to 48 KiB each) by
// global_load_lds_dwordx4.  Wave w owns k-step w % 4 of a stage's four and product w / 4: NT column tiles x MT row tiles; the
// four partial sums are added in order through LDS, where each wave then finds both sums of the results that it ends and
// stores.  A row's 16 chunks of 16 bytes sit at chunk ^ (row % 16), so that the 16 rows of a fragment read fall on 16 bank
// groups.  Rows past the weights' end are the last one again, columns of a tile past `cols` whatever lies in LDS: results that nobody stores.
// us, weights from memory, the two products on the kernels they get alone and the ops between them / this: 32 x 11008, K 4096
// 48.6 / 39.4 (180 MB: 4.6 TB/s), 64 x 11008 58.8 / 40.7, 32 x 5632, K 2048 27.2 / 11.9, 32 x 2816, K 1024 13.9 / 5.4; random
// sizes of up to 64 rows 2.0 times (74 of them, at least 1.14), of 65 to 128 rows and up to 8192 columns 2.05 (41, 1.28).
constexpr int gated_rows_stages(int mt, int nt) {
  const int stage = 16 * (mt + 2 * nt) * GR_KB;
  return 160 * 1024 / stage < 4 ? 160 * 1024 / stage : 4;
}
template <int MT, int NT> __global__ __launch_bounds__(512, 1) void gemm_gated_rows_kernel(GemmParams p, const void *up, int cols) {
  constexpr int KB = GR_KB, A_BYTES = 16 * MT * KB, W_BYTES = 16 * NT * KB, STAGE = A_BYTES + 2 * W_BYTES;
  constexpr int NST = gated_rows_stages(MT, NT);
  constexpr int NA = MT / 2, PER = NA + NT; // requests of 4 rows per wave and stage
  static_assert(NST >= 3 && 2 * NT * MT * 4096 <= NST * STAGE, "a ring, and room for the partial sums");
  __shared__ __align__(1024) char smem[NST * STAGE];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ks = wave & 3, mat = wave >> 2;
  const int r16 = lane & 15, g16 = lane >> 4;
  const int64_t n0 = (int64_t)blockIdx.x * cols;
  const int cols_in = (int)min((int64_t)cols, p.N - n0);
  const int64_t lda_b = p.lda * 2, ldb_b = p.ldb * 2;
  const int KT = (int)(p.K * 2 / KB);

  // requests: 2 per 8 rows of A, then cols / 4 per product, dealt to the waves in turn; behind the last one it is repeated, so
  // that every wave has as many to wait for
  uint32_t a_src[NA], w_src[NT];
  const char *w_ptr[NT];
  uint32_t w_dst[NT];
  {
    const int pos = lane & 15;
#pragma unroll
    for (int i = 0; i < NA; i++) {
      const int row = 4 * (8 * i + wave) + (lane >> 4);
      a_src[i] = (uint32_t)(min(row, (int)p.M - 1) * lda_b + ((pos ^ (row & 15)) << 4));
    }
    const int per = cols / 4;
#pragma unroll
    for (int i = 0; i < NT; i++) {
      const int q = min(8 * i + wave, 2 * per - 1), m = q >= per ? 1 : 0, row0 = 4 * (q - m * per), row = row0 + (lane >> 4);
      w_src[i] = (uint32_t)(min(row, cols_in - 1) * ldb_b + ((pos ^ (row & 15)) << 4));
      w_ptr[i] = reinterpret_cast<const char *>(m ? up : p.B) + n0 * ldb_b;
      w_dst[i] = (uint32_t)(A_BYTES + m * W_BYTES + row0 * KB);
    }
  }
  const char *a_ptr = reinterpret_cast<const char *>(p.A);
  // (the __restrict__ pointers give the requests and the fragment reads separate alias scopes: without them the
  // compiler makes every fragment read wait for all requests in flight)
  auto issue = [&](char *__restrict__ stage, int kt) {
#pragma unroll
    for (int i = 0; i < NA; i++)
      __builtin_amdgcn_global_load_lds((GCMI_GLB const void *)(a_ptr + (int64_t)kt * KB + a_src[i]),
                                       (GCMI_LDS void *)(stage + (8 * i + wave) * 1024), 16, 0, 0);
#pragma unroll
    for (int i = 0; i < NT; i++)
      __builtin_amdgcn_global_load_lds((GCMI_GLB const void *)(w_ptr[i] + (int64_t)kt * KB + w_src[i]),
                                       (GCMI_LDS void *)(stage + w_dst[i]), 16, 0, 0);
  };
  f32x4_t acc[NT][MT];
#pragma unroll
  for (int jt = 0; jt < NT; jt++)
#pragma unroll
    for (int it = 0; it < MT; it++)
      acc[jt][it] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  const uint32_t ld = (uint32_t)(r16 * KB + (((4 * ks + g16) ^ r16) << 4)), w_ld = (uint32_t)(A_BYTES + mat * W_BYTES) + ld;
  auto compute = [&](const char *__restrict__ st) {
    uint4 fa[MT], fb[NT];
#pragma unroll
    for (int it = 0; it < MT; it++)
      fa[it] = *reinterpret_cast<const uint4 *>(st + ld + it * 16 * KB);
#pragma unroll
    for (int jt = 0; jt < NT; jt++)
      fb[jt] = *reinterpret_cast<const uint4 *>(st + w_ld + jt * 16 * KB);
#pragma unroll
    for (int jt = 0; jt < NT; jt++)
#pragma unroll
      for (int it = 0; it < MT; it++)
        acc[jt][it] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, fb[jt]), __builtin_bit_cast(bf16x8_t, fa[it]),
                                                              acc[jt][it], 0, 0, 0);
  };
#pragma unroll
  for (int d = 0; d < NST - 1; d++)
    if (d < KT)
      issue(smem + d * STAGE, d);
  int slot = 0;
  for (int kt = 0; kt < KT; kt++) {
    // this wave's requests of stage kt have landed (those of the NST - 2 stages behind it may be in flight; near the
    // end fewer were issued, so everything is awaited); barrier: stage kt is visible, the slot of stage kt - 1 is free
    if (kt + NST - 2 < KT)
      asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NST - 2) * PER) : "memory");
    else
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    if (kt + NST - 1 < KT)
      issue(smem + (slot == 0 ? NST - 1 : slot - 1) * STAGE, kt + NST - 1);
    compute(smem + slot * STAGE);
    slot = slot == NST - 1 ? 0 : slot + 1;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); // this wave's reads of the stage are over before the next barrier
  }
  __syncthreads();
  // the k-steps' sums: [product][column tile][row tile][k-step][lane]
  f32x4_t *const red = reinterpret_cast<f32x4_t *>(smem);
#pragma unroll
  for (int jt = 0; jt < NT; jt++)
#pragma unroll
    for (int it = 0; it < MT; it++)
      red[(((mat * NT + jt) * MT + it) * 4 + ks) * 64 + lane] = acc[jt][it];
  __syncthreads();
  for (int t = wave; t < NT * MT; t += 8) {
    f32x4_t sum[2];
#pragma unroll
    for (int m = 0; m < 2; m++) {
      const f32x4_t *at = red + (m * NT * MT + t) * 256 + lane;
      sum[m] = at[0];
#pragma unroll
      for (int k = 1; k < 4; k++)
        sum[m] += at[64 * k];
    }
    const int m = 16 * (t % MT) + r16, col = 16 * (t / MT) + 4 * g16; // lane l holds columns 4 * (l / 16) .. + 3 of row l % 16
    if (m < p.M && col < cols_in)
      *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(p.C) + m * p.ldc + n0 + col) = gated_silu4(sum[0], sum[1]);
  }
}

// 32 * MI rows by 16 * NJ columns of C per workgroup
template <int MI, int NJ> __global__ __launch_bounds__(256, 1) void gemm_gated_kernel(GemmParams p, const void *up) {
  w4_body<2, true, MI, NJ, true>(p, up);
}

} // namespace gcmi

using namespace gcmi;

// rows x cols of C per workgroup; rows 0: the kernel that streams the weights
extern "C" int gcmi_launch_gemm_gated_tile(const GemmParams *pp, const void *up, int rows, int cols, hipStream_t stream) {
  GemmParams p = *pp;
  if (rows == 0) {
    const dim3 grid((unsigned)((p.N + cols - 1) / cols)), block(512);
#define GCMI_GATED_ROWS(NT)                                                                                           \
  if (p.M <= 32)                                                                                                      \
    hipLaunchKernelGGL((gemm_gated_rows_kernel<2, NT>), grid, block, 0, stream, p, up, cols);                         \
  else if (NT > 2 || p.M <= 64)                                                                                       \
    hipLaunchKernelGGL((gemm_gated_rows_kernel<4, NT>), grid, block, 0, stream, p, up, cols);                         \
  else                                                                                                                \
    hipLaunchKernelGGL((gemm_gated_rows_kernel<8, (NT > 2 ? 2 : NT)>), grid, block, 0, stream, p, up, cols)
    switch ((cols + 15) / 16) {
    case 1: GCMI_GATED_ROWS(1); break;
    case 2: GCMI_GATED_ROWS(2); break;
    case 3: GCMI_GATED_ROWS(3); break;
    default: GCMI_GATED_ROWS(4); break;
    }
#undef GCMI_GATED_ROWS
    return hipGetLastError() == hipSuccess ? 0 : 5;
  }
  p.group_m = 4;
  const dim3 grid((unsigned)(((p.M + rows - 1) / rows) * ((p.N + cols - 1) / cols))), block(256);
  if (rows == 128)
    hipLaunchKernelGGL((gemm_gated_kernel<4, 4>), grid, block, 0, stream, p, up);
  else if (rows == 192)
    hipLaunchKernelGGL((gemm_gated_kernel<6, 4>), grid, block, 0, stream, p, up);
  else if (cols == 64)
    hipLaunchKernelGGL((gemm_gated_kernel<8, 4>), grid, block, 0, stream, p, up);
  else if (cols == 96)
    hipLaunchKernelGGL((gemm_gated_kernel<8, 6>), grid, block, 0, stream, p, up);
  else
    hipLaunchKernelGGL((gemm_gated_kernel<8, 8>), grid, block, 0, stream, p, up);
  return hipGetLastError() == hipSuccess ? 0 : 5;
}

namespace {
// A tile's time in us, fitted to 174 random launches of 65 to 1000 rows with the weights from memory (rms error 3 to 11 %; past that,
// 75 sizes of 900 to 8192 rows are all ahead of two products and the ops between them, 1.05 to 7.7 times: 4096 x 11008, K 4096
// 596 / 569 us, 8192 x 5632, K 2048 347 / 319, 1500 x 11008, K 4096 343 / 220): a launch; per round of workgroups (one per compute unit) a start and an epilogue; per 128 of K its rounds and, as the clock and
// the memory system notice, its tiles per compute unit; per 2^20 results their store.
struct GatedTile {
  int rows, cols;
  double launch, round, group_round, group_load, mout;
};
const GatedTile GATED_TILES[] = {{128, 64, 4.3, 0.0, 0.95, 0.0, 1.5}, {192, 64, 3.5, 2.0, 1.12, 0.0, 1.3}, {256, 64, 2.6, 4.4, 1.26, 0.15, 0.5},
                                 {256, 96, 3.6, 8.4, 1.73, 0.31, 0.0}, {256, 128, 2.3, 10.0, 2.06, 0.25, 0.14}};
} // namespace

// silu(A . B^T) * (A . up^T): B and up [N,K], bf16 like A and C.  -1: not a call for these kernels (the caller runs its parts).
// dry: nothing is launched and the operands' addresses are not looked at; cfg != null receives what is chosen.
extern "C" int gcmi_launch_gemm_gated(const GemmParams *p, const void *up, hipStream_t stream, int dry, GemmTileConfig *cfg) {
  auto al16 = [](const void *q) { return (reinterpret_cast<uintptr_t>(q) & 15) == 0; };
  // few weights: the products alone are as long as a launch
  if (p->M < 1 || p->K < 128 || p->K % 8 != 0 || p->N % 4 != 0 || p->N * p->K < (int64_t)1 << 21 || p->lda % 8 != 0 || p->ldb % 8 != 0 ||
      p->ldc % 4 != 0 || p->lda * 2 * 256 >= (int64_t)1 << 31 || p->ldb * 2 * 256 >= (int64_t)1 << 31)
    return -1;
  if (!dry && !(al16(p->A) && al16(p->B) && al16(up) && (reinterpret_cast<uintptr_t>(p->C) & 7) == 0))
    return -1;
  const int n_cu = gcmi_num_cus();
  GemmTileConfig c{};
  c.split_k = 1, c.mfma_m = c.mfma_n = 16, c.mfma_k = 32;
  // Streaming: columns in fours, as few as fit one round of workgroups (more than 64 per compute unit: as few rounds as there are).
  const int64_t rounds = (p->N + 64 * (int64_t)n_cu - 1) / (64 * (int64_t)n_cu), per = (p->N + n_cu * rounds - 1) / (n_cu * rounds);
  const int cols = (int)((per + 3) / 4 * 4);
  if (p->K % 128 == 0 && p->K >= 512 && (p->M <= 64 || (p->M <= 128 && cols <= 32))) {
    c.kernel = GK_STREAM, c.bm = p->M <= 32 ? 32 : p->M <= 64 ? 64 : 128, c.bn = cols, c.kbytes = GR_KB, c.stages = gated_rows_stages(c.bm / 16, (cols + 15) / 16);
    c.waves_m = 1, c.waves_n = 2, c.wave_m = c.bm, c.wave_n = cols, c.group_m = 1, c.workgroups = (int32_t)((p->N + cols - 1) / cols);
    if (cfg)
      *cfg = c;
    return dry ? 0 : gcmi_launch_gemm_gated_tile(p, up, 0, cols, stream);
  }
  const GatedTile *tile = nullptr;
  double best = 0;
  int64_t tiles = 0;
  for (const GatedTile &t : GATED_TILES) {
    const int64_t n = ((p->M + t.rows - 1) / t.rows) * ((p->N + t.cols - 1) / t.cols);
    const double load = (double)n / n_cu, groups = (double)((p->K + 127) / 128);
    const double us = t.launch + t.round * ceil(load) + groups * (t.group_round * ceil(load) + t.group_load * load) +
                      t.mout * (double)p->M * (double)p->N / 1048576.0;
    if (!tile || us < best)
      tile = &t, best = us, tiles = n;
  }
  if (tiles > 0x7fffffff || (4 * tiles < n_cu && p->K > 1536))
    return -1;
  c.kernel = GK_WAVES4, c.bm = tile->rows, c.bn = tile->cols, c.kbytes = 64, c.stages = w4_ring_blocks<2, true>(tile->rows, 2 * tile->cols), c.group_m = 4, c.workgroups = (int32_t)tiles;
  c.waves_m = c.waves_n = 2, c.wave_m = tile->rows / 2, c.wave_n = tile->cols;
  if (cfg)
    *cfg = c;
  return dry ? 0 : gcmi_launch_gemm_gated_tile(p, up, tile->rows, tile->cols, stream);
}
