// Flash-Sinkhorn IFT backward with the plan in registers (scaled_bwd.h): a translation unit of its
// own so that it compiles in parallel with the general one, whose sweeps serve a group out of range.
//
// Bound by the latency of the solve's exchanges (two per iteration, about 2 us each with the sweep
// between them) and by the two passes of the cost gradient.  One multiply-add per element and sweep
// in place of a matrix product, a bias and an exponential: 16 heads of 389 tokens with bins and
// geometry, 7 fixed-point iterations: 229 us and 15 us for the bias matrix -> 85 us (no bias
// matrix); 2x8 heads of 768 tokens, 20 CG iterations: 180 -> 149 us.
#include "scaled_bwd.h"

namespace dfl {

template <typename T, bool GEN>
__global__ void __launch_bounds__(SB_NT) ift_scaled_kernel(IftBwdArgs a) {
  if (scaled_bwd<T, GEN>(a)) sinkhorn_bwd_general<T, 32, false, GEN>(fresh_args<IftBwdArgs>());
}

template <typename T, bool GEN>
static hipError_t launch_ift_t(const IftBwdArgs& a, size_t lds, hipStream_t stream, bool coop) {
  auto kern = ift_scaled_kernel<T, GEN>;
  hipError_t e = set_lds_limit((const void*)kern, lds);
  if (e != hipSuccess) return e;
  dim3 grid(grid_blocks(a.B * a.H, a.G)), block(SB_NT);
  IftBwdArgs copy = a;
  if (coop) {
    void* args[] = {&copy};
    return hipLaunchCooperativeKernel((const void*)kern, grid, block, args, (unsigned)lds, stream);
  }
  hipLaunchKernelGGL(kern, grid, block, lds, stream, copy);
  return hipGetLastError();
}

constexpr size_t IFT_STATIC = 1024;  // static LDS of the register form and the general backward, rounded up

bool sinkhorn_bwd_reg_n(int N, int G) { return reg_fits(N, G); }

bool sinkhorn_bwd_reg_fits(int N, int DP, int G, size_t lds_general, size_t limit) {
  return DP == 32 && reg_fits(N, G) && ift_lds_bytes(N, G) + IFT_STATIC <= limit && lds_general + IFT_STATIC <= limit;
}

hipError_t launch_sinkhorn_bwd_reg(const IftBwdArgs& a, bool bf16_in, size_t lds_general, hipStream_t stream, bool coop) {
  const bool gen = (a.bins8 && a.pos_w) || (a.x && a.w_dist);
  const size_t lds = std::max(ift_lds_bytes(a.N, a.G), lds_general);
  if (bf16_in)
    return gen ? launch_ift_t<bf16, true>(a, lds, stream, coop) : launch_ift_t<bf16, false>(a, lds, stream, coop);
  return gen ? launch_ift_t<float, true>(a, lds, stream, coop) : launch_ift_t<float, false>(a, lds, stream, coop);
}

}  // namespace dfl
