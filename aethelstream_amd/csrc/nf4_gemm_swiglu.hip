// nf4_gemm_swiglu.hip - launches of the SwiGLU-fused forward GEMM
// (nf4_gemm_core.hpp).
#include "nf4_gemm_core.hpp"

namespace nf4s {

int32_t launch_swiglu(GroupedArgs &ga, bool dq, bool batch, hipStream_t s) {
  const LaunchPlan p = plan_launch(ga.base.M, ga.tiles_o, ga.base.R / kStep, batch ? 4 : 2, 0);
  const int64_t T = apply_plan(ga, p, ga.tiles_o, nullptr);
  if (T < 0) return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "too many tiles");
  with_kmt(p.kmt, [&](auto K) {
    constexpr int kmt = decltype(K)::value;
    const dim3 grid(launch_grid(kmt, T)), block(kGemmThreads);
    if (batch && dq)
      hipLaunchKernelGGL((nf4_gemm_swiglu_kernel<kmt, FwdBatchProducer<true>>), grid, block, 0, s,
                         ga);
    else if (batch)
      hipLaunchKernelGGL((nf4_gemm_swiglu_kernel<kmt, FwdBatchProducer<false>>), grid, block, 0, s,
                         ga);
    else if (dq)
      hipLaunchKernelGGL((nf4_gemm_swiglu_kernel<kmt, FwdProducer<true>>), grid, block, 0, s, ga);
    else
      hipLaunchKernelGGL((nf4_gemm_swiglu_kernel<kmt, FwdProducer<false>>), grid, block, 0, s, ga);
  });
  return check_launch("nf4_gemm_swiglu");
}

}  // namespace nf4s
