// The 4-wave kernels of 128 to 256 rows by 128 or 192 columns (gemm_tile256.hpp) for bf16 operands, B stored [N,K].
#include "gemm_tile256.hpp"

using namespace gcmi;

extern "C" int gcmi_launch_tall_bf16_nt(const GemmParams *p, int rows, int cols, unsigned grid_x, unsigned grid_y, hipStream_t stream) {
  return launch_tall<true, 2>(*p, rows, cols, dim3(grid_x, grid_y), stream);
}
