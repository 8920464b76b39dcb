// Split-precision instances of the direct-stage NT GEMM (ngemm_kernel.hpp).
#include "ngemm_kernel.hpp"

namespace tci {

namespace {
template <int PREC>
void launch_p(int shape, dim3 g, const Task* tasks, const NSeg* segs, int64_t J0, const float* sc, hipStream_t st,
              int remap) {
  switch (shape) {
    case N128:
      hipLaunchKernelGGL((ngemm_kernel<S16T<PREC>, 2, 2, 1, 4, 4, 2, 2>), g, dim3(256), 0, st, tasks, segs, J0, sc, remap);
      break;
    case N128x192:
      hipLaunchKernelGGL((ngemm_kernel<S16T<PREC>, 2, 2, 1, 4, 6, 2, 2>), g, dim3(256), 0, st, tasks, segs, J0, sc, remap);
      break;
    case N192:
      hipLaunchKernelGGL((ngemm_kernel<S16T<PREC>, 2, 4, 1, 6, 3, 3, 2>), g, dim3(512), 0, st, tasks, segs, J0, sc, remap);
      break;
    case N64:
      hipLaunchKernelGGL((ngemm_kernel<S16T<PREC>, 2, 2, 1, 2, 2, 2, 4>), g, dim3(256), 0, st, tasks, segs, J0, sc, remap);
      break;
    case N32K4:
      hipLaunchKernelGGL((ngemm_kernel<S16T<PREC>, 1, 1, 4, 2, 2, 2, 2>), g, dim3(256), 0, st, tasks, segs, J0, sc, remap);
      break;
    case N256:
      hipLaunchKernelGGL((ngemm_kernel<S32T<PREC>, 2, 4, 1, 4, 2, 2, 2>), g, dim3(512), 0, st, tasks, segs, J0, sc, remap);
      break;
    default: throw Error(TCI_ERR_ARG, "no split NT GEMM tile of this shape");
  }
}
}  // namespace

void launch_ngemm16(int precision, int shape, const Task* tasks, const NSeg* segs, int64_t ntasks, int64_t J0,
                    const float* scales, hipStream_t st, int remap) {
  if (ntasks <= 0) return;
  TCI_REQUIRE(ntasks < ((int64_t)1 << 31), "too many gemm tasks");
  const dim3 g((unsigned)ntasks);
  if (precision == TCI_SIGMA_BF16X3) launch_p<TCI_SIGMA_BF16X3>(shape, g, tasks, segs, J0, scales, st, remap);
  else launch_p<TCI_SIGMA_FP16X3>(shape, g, tasks, segs, J0, scales, st, remap);
  TCI_HIP(hipGetLastError());
}

}  // namespace tci
