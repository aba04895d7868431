// nf4_gemm_fwd.hip - launches of the tiled forward GEMM (nf4_gemm_core.hpp).
#include "nf4_gemm_core.hpp"

namespace nf4s {

template <class Producer>
static int32_t launch(GroupedArgs &ga, hipStream_t s, void *ws, int64_t ws_bytes) {
  const LaunchPlan p = plan_launch(ga.base.M, ga.tiles_o, ga.base.R / kStep, Producer::kUnroll,
                                   ws != nullptr ? ws_bytes : 0);
  const int64_t U = apply_plan(ga, p, ga.tiles_o, ws);
  if (U == 0) return NF4S_OK;
  if (U < 0) return fail(NF4S_ERR_UNSUPPORTED_SHAPE, "too many tiles");
  int32_t rc = NF4S_OK;
  with_kmt(p.kmt, [&](auto K) {
    constexpr int kmt = decltype(K)::value;
    hipLaunchKernelGGL((nf4_gemm_fwd_kernel<kmt, Producer>), dim3(launch_grid(kmt, U)),
                       dim3(kGemmThreads), 0, s, ga);
    rc = check_launch("nf4_gemm_fwd");
    if (rc == NF4S_OK && ga.splits > 1) {
      hipLaunchKernelGGL((nf4_gemm_fixup_kernel<kmt, false>),
                         dim3((uint32_t)(p.split.tail_tiles * fixup_blocks_per_tile(kmt))),
                         dim3(kGemmThreads), 0, s, ga);
      rc = check_launch("nf4_gemm_fixup");
    }
  });
  return rc;
}

int32_t launch_fwd(GroupedArgs &ga, bool dq, bool batch, hipStream_t s, void *ws,
                   int64_t ws_bytes) {
  if (batch)
    return dq ? launch<FwdBatchProducer<true>>(ga, s, ws, ws_bytes)
              : launch<FwdBatchProducer<false>>(ga, s, ws, ws_bytes);
  return dq ? launch<FwdProducer<true>>(ga, s, ws, ws_bytes)
            : launch<FwdProducer<false>>(ga, s, ws, ws_bytes);
}

}  // namespace nf4s
