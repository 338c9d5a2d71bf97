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
  const bool pair = tile128_in_pairs(es, rows, cols, p->K, p->splits, (int64_t)grid_x * grid_y);
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
