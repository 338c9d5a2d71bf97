// bf16 x bf16 -> f32 GEMMs: the MFMA tile kernels (gemm_tile256.hpp, gemm_tile128.hpp) and those for a short A:
// gemm_rows32.hpp streams wide weights past up to 128 rows, gemm_few_rows.hpp takes up to 256 rows in one launch where a
// round of its tiles holds them, gemm_skinny.hpp [N,K] weights where a caller's slice count asks for it and the shapes
// the others do not take.
#include "gemm_rows32.hpp"
#include "gemm_skinny.hpp"

extern "C" int gcmi_launch_few_rows(const gcmi::GemmParams *p, int es, hipStream_t stream, int dry, gcmi::GemmTileConfig *cfg,
                                    int slices); // gemm_few_rows.hip

// Floats of workspace that the kernels behind the few-row one would use for this call; *optional: see the query below.
static int64_t slices_want(const gcmi::GemmParams *p, bool *optional) {
  int64_t want = 0;
  *optional = false;
  if (gcmi::launch_skinny_nt(p, nullptr, &want) >= 0)
    return want;
  gcmi::launch_tile256<2>(p, nullptr, &want, nullptr, optional);
  *optional = *optional || p->K % (256 / 2) != 0;
  return want;
}

// A call of few rows.  One with a long K is left to K slices where another kernel has them and two of them at least fit the
// workspace.
static int launch_few(const gcmi::GemmParams *p, hipStream_t stream, bool dry, gcmi::GemmTileConfig *cfg) {
  const int rc = gcmi_launch_few_rows(p, 2, stream, dry, cfg, 1);
  if (rc >= 0 || gcmi_launch_few_rows(p, 2, nullptr, 1, nullptr, 0) < 0)
    return rc;
  bool optional;
  if (p->partial && p->partial_cap >= 2 * p->M * p->N && slices_want(p, &optional) > 0)
    return -1;
  return gcmi_launch_few_rows(p, 2, stream, dry, cfg, 0);
}

extern "C" int gcmi_launch_gemm_bf16(const gcmi::GemmParams *p, hipStream_t stream) {
  int rc = gcmi::launch_rows32(p, stream);
  if (rc >= 0)
    return rc;
  rc = launch_few(p, stream, false, nullptr);
  if (rc >= 0)
    return rc;
  rc = gcmi::launch_skinny_nt(p, stream);
  if (rc >= 0)
    return rc;
  return gcmi::launch_tile256<2>(p, stream);
}

// Floats of workspace (GemmParams::partial) the launch above would use for this call: 0 when K is not sliced.
// *optional: the call is one that has to run without as well (in one pass, the sums in another order): a K with an
// incomplete ring group, which the tile kernels slice like any other K, a call of few rows whose slices are only the faster
// way, or one that is sliced only since there are tiles of more than 128 rows.  No entry point may refuse these under stream
// capture, as it does the others with a K of whole groups.
extern "C" int64_t gcmi_launch_gemm_bf16_workspace(const gcmi::GemmParams *p, int *optional) {
  int64_t want = 0;
  *optional = 0;
  if (gcmi::launch_rows32(p, nullptr, &want) >= 0)
    return want;
  if (gcmi_launch_few_rows(p, 2, nullptr, 1, nullptr, 1) >= 0)
    return 0;
  bool one_pass_too = false;
  want = slices_want(p, &one_pass_too);
  *optional = one_pass_too || gcmi_launch_few_rows(p, 2, nullptr, 1, nullptr, 0) >= 0;
  return want;
}

// what the launch above would choose (nothing is launched)
extern "C" int gcmi_launch_gemm_bf16_config(const gcmi::GemmParams *p, gcmi::GemmTileConfig *cfg) {
  if (gcmi::launch_rows32(p, (hipStream_t)-1, nullptr, cfg) >= 0)
    return 0;
  if (launch_few(p, nullptr, true, cfg) >= 0)
    return 0;
  if (gcmi::launch_skinny_nt(p, (hipStream_t)-1, nullptr, cfg) >= 0)
    return 0;
  return gcmi::launch_tile256<2>(p, (hipStream_t)-1, nullptr, cfg);
}

// Scratch of the entry point that allocates nothing (gcmi_gemm_bf16_noalloc): the partial sums of K-sliced calls.
// Each device the library runs on holds its own copy until the process ends.  `scratch` is only a host-side
// stand-in here: its device address is asked for once per device and kept.
static constexpr size_t GCMI_NOALLOC_SCRATCH_BYTES = (size_t)32 << 20;
static __device__ __align__(256) unsigned char scratch[GCMI_NOALLOC_SCRATCH_BYTES];

extern "C" int gcmi_noalloc_scratch(void **ptr, size_t *bytes) {
  static void *dev_ptr[64];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= 64)
    return 5;
  void *q = __atomic_load_n(&dev_ptr[dev], __ATOMIC_ACQUIRE);
  if (!q) {
    if (hipGetSymbolAddress(&q, HIP_SYMBOL(scratch)) != hipSuccess || !q)
      return 5;
    __atomic_store_n(&dev_ptr[dev], q, __ATOMIC_RELEASE); // the same value from every thread that gets here
  }
  *ptr = q;
  *bytes = GCMI_NOALLOC_SCRATCH_BYTES;
  return 0;
}
