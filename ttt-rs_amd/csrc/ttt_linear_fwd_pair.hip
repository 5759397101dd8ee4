// The f32 TTT-Linear forward on two workgroups per unit as a translation unit of its own (it compiles beside ttt_api.hip).
#include "ttt_linear_fwd_pair.hip.h"

namespace ttt {

template <int D, bool CKPT, bool REST = false>
static hipError_t launch(const LinearFwdArgs& a, const LinearPairArgs& pa, hipStream_t s) {
  const unsigned units = (unsigned)(a.B * a.H);
  hipLaunchKernelGGL((ttt_linear_fwd_pair_clear_kernel<D>), dim3((units + 127) / 128), dim3(128), 0, s, a.W_out, (int)units);
  hipLaunchKernelGGL((ttt_linear_fwd_pair_kernel<D, CKPT, REST>), dim3((units + 7) / 8 * 16), dim3(64 * (D / 16 + 2)), 0, s, a, pa);
  if constexpr (REST)
    hipLaunchKernelGGL((ttt_linear_fwd_redo_rest_kernel<D>), dim3(units), dim3(64 * (D / 16)), 0, s, a, pa.rest);
  else
    hipLaunchKernelGGL((ttt_linear_fwd_redo_kernel<D, CKPT>), dim3(units), dim3(64 * (D / 16 + 1)), 0, s, a);
  return hipGetLastError();
}

hipError_t launch_linear_fwd_pair(int head_dim, const LinearFwdArgs& a, const LinearPairArgs& pa, hipStream_t s) {
  const bool ckpt = a.W_ckpt != nullptr;
  if (pa.rest > 0) return head_dim == 64 ? launch<64, false, true>(a, pa, s) : launch<32, false, true>(a, pa, s);
  if (head_dim == 64) return ckpt ? launch<64, true>(a, pa, s) : launch<64, false>(a, pa, s);
  return ckpt ? launch<32, true>(a, pa, s) : launch<32, false>(a, pa, s);
}

}  // namespace ttt
