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
  // Runs of tiles for the XCDs give each a few rows and many columns; with few columns of tiles an XCD needs most of B either way, and
  // in the hardware's order all of them read it side by side.  8-bit operands, K of 1024 and more, a number of tiles that is no multiple
  // of 8, us, runs / hardware's order: up to 20 columns of tiles 2056 x 2208, K 1104 17.2 / 16.0, 1693 x 2384, K 1120 16.3 / 15.1,
  // 3309 x 1824, K 2160 27.0 / 25.4, 3551 x 1840, K 2464 30.1 / 28.4 (20 sizes 0.989 to 1.086 times, 1.02 on the average); past
  // that 1322 x 5696, K 1440 19.9 / 21.8, 1457 x 4960, K 2336 29.5 / 33.4, 2224 x 2912, K 2368 26.8 / 28.2; with a shorter K 5439 x 736,
  // K 480 9.0 / 10.0, 4529 x 1392, K 720 0.98 times.
  if (es == 1 && grid_x % 8 != 0 && grid_y == 1 && p->K >= 1024 && (p->N + 127) / 128 <= 20)
    hipLaunchKernelGGL((gemm_tile128_kernel<false, 1, false>), grid, block, 0, stream, *p);
  else if (es == 1)
    hipLaunchKernelGGL((gemm_tile128_kernel<false, 1>), grid, block, 0, stream, *p);
  else if (p->trans_b)
    hipLaunchKernelGGL((gemm_tile128_kernel<true, 2>), grid, block, 0, stream, *p);
  else
    hipLaunchKernelGGL((gemm_tile128_kernel<false, 2>), grid, block, 0, stream, *p);
  return hipGetLastError() == hipSuccess ? 0 : 5;
}
}
