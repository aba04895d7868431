// nf4_gemm_dgrad.hip - launches of the input-gradient GEMM
// (nf4_gemm_core.hpp).
#include "nf4_gemm_core.hpp"

namespace nf4s {

template <class Producer>
static int32_t launch(GroupedArgs &ga, int64_t nsteps, hipStream_t s, void *ws,
                      int64_t ws_bytes) {
  const LaunchPlan p = plan_launch(ga.base.M, ga.base.tiles_o, nsteps, Producer::kUnroll,
                                   ws != nullptr ? ws_bytes : 0);
  const int64_t U = apply_plan(ga, p, ga.base.tiles_o, ws);
  if (U == 0) return NF4S_OK;
  if (U < 0) return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "too many tiles");
  int32_t rc = NF4S_OK;
  with_kmt(p.kmt, [&](auto K) {
    constexpr int kmt = decltype(K)::value;
    const dim3 grid(launch_grid(kmt, U)), block(kGemmThreads);
    if (ga.splits > 1)
      hipLaunchKernelGGL((nf4_gemm_dgrad_kernel<kmt, Producer, true>), grid, block, 0, s, ga);
    else
      hipLaunchKernelGGL((nf4_gemm_dgrad_kernel<kmt, Producer, false>), grid, block, 0, s, ga);
    rc = check_launch("nf4_gemm_dgrad");
    if (rc == NF4S_OK && ga.splits > 1) {
      hipLaunchKernelGGL((nf4_gemm_fixup_kernel<kmt, true>),
                         dim3((uint32_t)(p.split.tail_tiles * fixup_blocks_per_tile(kmt))), block,
                         0, s, ga);
      rc = check_launch("nf4_gemm_fixup");
    }
  });
  return rc;
}

int32_t launch_dgrad(GroupedArgs &ga, int64_t nsteps, bool dq, bool batch, hipStream_t s,
                     void *ws, int64_t ws_bytes) {
  if (batch)
    return dq ? launch<DgradBatchProducer<true>>(ga, nsteps, s, ws, ws_bytes)
              : launch<DgradBatchProducer<false>>(ga, nsteps, s, ws, ws_bytes);
  return dq ? launch<DgradProducer<true>>(ga, nsteps, s, ws, ws_bytes)
            : launch<DgradProducer<false>>(ga, nsteps, s, ws, ws_bytes);
}

}  // namespace nf4s
