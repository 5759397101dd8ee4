// The bf16 TTT-Linear forward with the waves of a unit in roles, as a translation unit of its own (it compiles beside ttt_api.hip).
#include "ttt_linear_fwd_roles.hip.h"

namespace ttt {

template <int D, bool TWO>
static hipError_t launch(const LinearFwdArgs* probs, unsigned ny, int cus, int rest, hipStream_t s) {
  Problems<LinearFwdArgs> P;
  bool states = false, factors = false;
  for (unsigned y = 0; y < ny; ++y) {
    P.p[y] = probs[y];
    (probs[y].ckpt_packed == kCkptFactors ? factors : states) |= probs[y].W_ckpt != nullptr;
  }
  const dim3 grid((unsigned)(probs[0].B * probs[0].H), ny), block(64 * 5);
  if (rest > 0)
    hipLaunchKernelGGL((ttt_linear_fwd_roles_kernel<D, 0, TWO, true>), grid, block, 0, s, P, cus, rest);
  else if (factors)
    hipLaunchKernelGGL((ttt_linear_fwd_roles_kernel<D, 2, TWO, false>), grid, block, 0, s, P, cus, rest);
  else if (states)
    hipLaunchKernelGGL((ttt_linear_fwd_roles_kernel<D, 1, TWO, false>), grid, block, 0, s, P, cus, rest);
  else
    hipLaunchKernelGGL((ttt_linear_fwd_roles_kernel<D, 0, TWO, false>), grid, block, 0, s, P, cus, rest);
  return hipGetLastError();
}

hipError_t launch_linear_fwd_roles_form(int head_dim, const LinearFwdArgs& a, const FusedInputsArgs& fi, int cus, hipStream_t s) {
  const dim3 grid((unsigned)(a.B * a.H)), block(64 * 6);
  if (head_dim == 64)
    hipLaunchKernelGGL((ttt_linear_fwd_roles_form_kernel<64, false>), grid, block, 0, s, a, fi, cus);
  else if ((long)a.B * a.H <= cus)
    hipLaunchKernelGGL((ttt_linear_fwd_roles_form_kernel<32, false>), grid, block, 0, s, a, fi, cus);
  else
    hipLaunchKernelGGL((ttt_linear_fwd_roles_form_kernel<32, true>), grid, block, 0, s, a, fi, cus);
  return hipGetLastError();
}

hipError_t launch_linear_fwd_roles(int head_dim, const LinearFwdArgs* probs, unsigned ny, int cus, int rest, hipStream_t s) {
  if (head_dim == 64) return launch<64, false>(probs, ny, cus, rest, s);
  return (long)probs[0].B * probs[0].H * ny > cus ? launch<32, true>(probs, ny, cus, rest, s) : launch<32, false>(probs, ny, cus, rest, s);
}

}  // namespace ttt
