// The 4-wave kernels of 128 to 256 rows by 128 columns (gemm_tile256.hpp) for 8-bit operands.
#include "gemm_tile256.hpp"

using namespace gcmi;

extern "C" int gcmi_launch_tall_int8(const GemmParams *p, int rows, int cols, unsigned grid_x, unsigned grid_y, hipStream_t stream) {
  return launch_tall<false, 1>(*p, rows, cols, dim3(grid_x, grid_y), stream);
}
