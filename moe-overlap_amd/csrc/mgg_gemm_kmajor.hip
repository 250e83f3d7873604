// Launches of the K-major 256x256 kernel (mgg_gemm_kmajor.h).
#include "mgg_gemm_kmajor.h"

namespace mgg {
namespace {

template <class T>
int launch_typed(int epilogue, const GemmParams& p, int workers, hipStream_t stream) {
  const dim3 grid(workers), block(kKmThreads);
  switch (epilogue) {
    case kEpiNone:
      hipLaunchKernelGGL((grouped_gemm_kmajor_kernel<T, kEpiNone>), grid, block, 0, stream, p);
      return MGG_OK;
    case kEpiGelu:
      hipLaunchKernelGGL((grouped_gemm_kmajor_kernel<T, kEpiGelu>), grid, block, 0, stream, p);
      return MGG_OK;
    case kEpiSwiglu:
      hipLaunchKernelGGL((grouped_gemm_kmajor_kernel<T, kEpiSwiglu>), grid, block, 0, stream, p);
      return MGG_OK;
    default: return set_error(MGG_ERR_INVALID, "unknown epilogue");
  }
}

}  // namespace

int launch_kmajor_256(int dtype, int epilogue, const GemmParams& p, int workers, hipStream_t stream) {
  return dtype == (MGG_DTYPE_BF16 | MGG_B_KMAJOR) ? launch_typed<Bf16K>(epilogue, p, workers, stream)
                                                  : launch_typed<F16K>(epilogue, p, workers, stream);
}

}  // namespace mgg
