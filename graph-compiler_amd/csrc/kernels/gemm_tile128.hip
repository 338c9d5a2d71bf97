// The kernel of gemm_tile128.hpp, in a translation unit of its own, and the choice between it and the 4-wave kernels with the
// hand-placed loop.
#include "gemm_tile256.hpp"
#include "gemm_tile128.hpp"

using namespace gcmi;

extern "C" {
int gcmi_launch_tall_bf16(const GemmParams *p, int rows, int cols, unsigned grid_x, unsigned grid_y, hipStream_t stream);
int gcmi_launch_tall_bf16_nt(const GemmParams *p, int rows, int cols, unsigned grid_x, unsigned grid_y, hipStream_t stream);
int gcmi_launch_tall_int8(const GemmParams *p, int rows, int cols, unsigned grid_x, unsigned grid_y, hipStream_t stream);

// es: bytes of an element of A; rows, cols: the tile's, 128 / 192 / 256 by 128 or 256 by 192
int gcmi_launch_tile128(const GemmParams *p, int es, int rows, int cols, unsigned grid_x, unsigned grid_y, hipStream_t stream) {
  // Two 128 x 128 tiles per compute unit only where there are more than a round of them, or two groups of K or less, which are
  // set-up and epilogue mostly.  Else the hand-placed loop with its deeper ring, the whole LDS to itself, us, two per unit / this,
  // weights from memory: 1000 x 4096, K 4096 [N,K] 48.2 / 37.2, 2048^3 27.8 / 23.7, 1422 x 2384, K 1280 [N,K] 16.3 / 12.9, 1086 x 144,
  // K 272 7.6 / 7.4, 8-bit 1024 x 4096, K 4096 31.5 / 26.9; but 746 x 944, K 160 7.4 / 7.6, 8-bit 1425 x 1168, K 208 7.9 / 8.3, and in more
  // than a round 2498 x 2544, K 512 13.3 / 14.2.
  const bool pair = rows == 128 && cols == 128 &&
                    ((int64_t)grid_x * grid_y > gcmi_num_cus() || p->K * es <= 512 * (int64_t)(p->splits > 1 ? p->splits : 1));
  if (!pair)
    return es == 1 ? gcmi_launch_tall_int8(p, rows, cols, grid_x, grid_y, stream)
           : p->trans_b ? gcmi_launch_tall_bf16_nt(p, rows, cols, grid_x, grid_y, stream)
                        : gcmi_launch_tall_bf16(p, rows, cols, grid_x, grid_y, stream);
  const dim3 grid(grid_x, grid_y), block(256);
  if (es == 1)
    hipLaunchKernelGGL((gemm_tile128_kernel<false, 1>), grid, block, 0, stream, *p);
  else if (p->trans_b)
    hipLaunchKernelGGL((gemm_tile128_kernel<true, 2>), grid, block, 0, stream, *p);
  else
    hipLaunchKernelGGL((gemm_tile128_kernel<false, 2>), grid, block, 0, stream, *p);
  return hipGetLastError() == hipSuccess ? 0 : 5;
}
}
