// The TTT-MLP forward with several hidden layers as a translation unit of its own (it compiles beside ttt_api.hip).
#include "ttt_mlpn_fwd.hip.h"

namespace ttt {

template <class T, int D, int NL>
static hipError_t launch(const MlpNFwdArgs& a, hipStream_t s) {
  constexpr auto kern = ttt_mlpn_fwd_kernel<T, D, NL>;
  constexpr int bytes = (int)MlpNLds<D, NL>::BYTES;
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(kern, dim3((unsigned)(a.B * a.H)), dim3(512), bytes, s, a);
  return hipGetLastError();
}

template <class T>
static hipError_t launch(int head_dim, int n_hidden, const MlpNFwdArgs& a, hipStream_t s) {
  if (head_dim == 64) return launch<T, 64, 2>(a, s);
  switch (n_hidden) {
    case 2: return launch<T, 32, 2>(a, s);
    case 3: return launch<T, 32, 3>(a, s);
    default: return launch<T, 32, 4>(a, s);
  }
}

hipError_t launch_mlpn_fwd(bool f32, int head_dim, int n_hidden, const MlpNFwdArgs& a, hipStream_t s) {
  return f32 ? launch<F32>(head_dim, n_hidden, a, s) : launch<BF16>(head_dim, n_hidden, a, s);
}

}  // namespace ttt
