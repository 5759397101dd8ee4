// The register-resident TTT-MLP backward as a translation unit of its own (it compiles beside ttt_api.hip).
#include "ttt_mlp_bwd_rp.hip.h"

namespace ttt {

template <int D>
static hipError_t launch(const MlpBwdRpArgs& a, hipStream_t s) {
  constexpr auto kern = ttt_mlp_bwd_rp_kernel<D>;
  constexpr int bytes = MlpRpLds<D>::BYTES;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return e;
  // two workgroups per unit: workgroups b and b + 8 of every 16 share a unit
  const unsigned units = (unsigned)(a.B * a.H), grid = a.role == 2 ? (units + 7) / 8 * 16 : units;
  hipLaunchKernelGGL(kern, dim3(grid), dim3(512), bytes, s, a);
  return hipGetLastError();
}

hipError_t launch_mlp_bwd_rp(int head_dim, const MlpBwdRpArgs& a, hipStream_t s) {
  return head_dim == 32 ? launch<32>(a, s) : head_dim == 64 ? launch<64>(a, s) : launch<96>(a, s);
}

}  // namespace ttt
