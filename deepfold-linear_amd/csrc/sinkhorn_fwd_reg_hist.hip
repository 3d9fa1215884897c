// Flash-Sinkhorn forward with register storage, the forms that record the potentials of every
// half-iteration (sinkhorn_fwd_kernel.h, FWD_HIST_REG and FWD_BAL_REG).
#include "sinkhorn_fwd_kernel.h"

namespace dfl {

hipError_t launch_sinkhorn_fwd_reg_hist(const SinkFwdArgs& a, bool bf16_in, int DP, size_t lds, hipStream_t stream,
                                        bool coop) {
  if (!a.hist) return hipErrorInvalidValue;
  if (a.balanced) return launch_fwd_dt<false, FWD_BAL_REG, true>(a, bf16_in, DP, lds, stream, coop);
  const bool gen = (a.bins8 && a.pos_w) || (a.x && a.w_dist);
  return gen ? launch_fwd_dt<false, FWD_HIST_REG, true>(a, bf16_in, DP, lds, stream, coop)
             : launch_fwd_dt<false, FWD_HIST_REG, false>(a, bf16_in, DP, lds, stream, coop);
}

}  // namespace dfl
