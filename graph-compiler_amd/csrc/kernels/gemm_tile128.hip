// The kernels of gemm_tile128.hpp, in a translation unit of their own.
#include "gemm_tile256.hpp"
#include "gemm_tile128.hpp"

using namespace gcmi;

// es: bytes of an element of A; rows: the tile's, 128, 192 or 256
extern "C" int gcmi_launch_tile128(const GemmParams *p, int es, int rows, unsigned grid_x, unsigned grid_y, hipStream_t stream) {
  const dim3 grid(grid_x, grid_y), block(256);
#define GCMI_T128(TB, ES)                                                                                             \
  if (rows == 256)                                                                                                    \
    hipLaunchKernelGGL((gemm_tall_kernel<TB, ES, 8>), grid, block, 0, stream, *p);                                 \
  else if (rows == 192)                                                                                               \
    hipLaunchKernelGGL((gemm_tall_kernel<TB, ES, 6>), grid, block, 0, stream, *p);                                 \
  else                                                                                                                \
    hipLaunchKernelGGL((gemm_tile128_kernel<TB, ES>), grid, block, 0, stream, *p);
  if (es == 1) {
    GCMI_T128(false, 1)
  } else if (p->trans_b) {
    GCMI_T128(true, 2)
  } else {
    GCMI_T128(false, 2)
  }
#undef GCMI_T128
  return hipGetLastError() == hipSuccess ? 0 : 5;
}
