// The kernels of gemm_few_rows.hpp, in a translation unit of their own.
#include "gemm_few_rows.hpp"

// es: bytes of an element of A (2: bf16, 1: 8-bit).  dry: nothing is launched.  slices: see launch_few_rows.  -1: not this
// kernel's call.
extern "C" int gcmi_launch_few_rows(const gcmi::GemmParams *p, int es, hipStream_t stream, int dry, gcmi::GemmTileConfig *cfg, int slices) {
  return es == 2 ? gcmi::launch_few_rows<2>(p, stream, dry != 0, cfg, slices != 0)
                 : gcmi::launch_few_rows<1>(p, stream, dry != 0, cfg, false);
}
