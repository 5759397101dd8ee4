// The TTT-MLP forward with several hidden layers as a translation unit of its own (it compiles beside ttt_api.hip).
#include "ttt_mlpn_fwd.hip.h"

namespace ttt {

template <class T, int D, int NL>
static hipError_t launch(bool pair, const MlpNFwdArgs& a, hipStream_t s) {
  constexpr int bytes = (int)MlpNLds<D, NL>::BYTES;
  const unsigned units = (unsigned)(a.B * a.H);
  const auto launch_lds = [&](auto kern, unsigned blocks, const MlpNFwdArgs& args) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e == hipSuccess) hipLaunchKernelGGL(kern, dim3(blocks), dim3(512), bytes, s, args);
    return e;
  };
  MlpNFwdArgs one = a;
  one.only_lost = pair ? 1 : 0;
  if (pair) {
    hipLaunchKernelGGL((ttt_mlpn_fwd_clear_kernel<D, NL>), dim3(units), dim3(MlpNPair<D, NL>::FL_WORDS), 0, s, a);
    const hipError_t e = launch_lds(ttt_mlpn_fwd_pair_kernel<T, D, NL>, (units + 7) / 8 * 16, a);
    if (e != hipSuccess) return e;
  }
  const hipError_t e = launch_lds(ttt_mlpn_fwd_kernel<T, D, NL>, units, one);
  if (e != hipSuccess) return e;
  return hipGetLastError();
}

template <class T>
static hipError_t launch(int head_dim, int n_hidden, bool pair, const MlpNFwdArgs& a, hipStream_t s) {
  if (head_dim == 64) return launch<T, 64, 2>(pair, a, s);
  switch (n_hidden) {
    case 2: return launch<T, 32, 2>(pair, a, s);
    case 3: return launch<T, 32, 3>(pair, a, s);
    default: return launch<T, 32, 4>(pair, a, s);
  }
}

hipError_t launch_mlpn_fwd(bool f32, int head_dim, int n_hidden, bool pair, const MlpNFwdArgs& a, hipStream_t s) {
  return f32 ? launch<F32>(head_dim, n_hidden, pair, a, s) : launch<BF16>(head_dim, n_hidden, pair, a, s);
}

}  // namespace ttt
