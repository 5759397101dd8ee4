// The register-resident TTT-MLP backward at head_dim 32 and 64 as a translation unit of its own (it compiles beside
// ttt_api.hip); head_dim 96 is ttt_mlp_bwd_rp_d96.hip.
#include "ttt_mlp_bwd_rp.hip.h"

namespace ttt {

hipError_t launch_mlp_bwd_rp_d96(const MlpBwdRpArgs& a, hipStream_t s);  // ttt_mlp_bwd_rp_d96.hip

hipError_t launch_mlp_bwd_rp(int head_dim, const MlpBwdRpArgs& a, hipStream_t s) {
  return head_dim == 32 ? launch_mlp_bwd_rp_d<32>(a, s) : head_dim == 64 ? launch_mlp_bwd_rp_d<64>(a, s) : launch_mlp_bwd_rp_d96(a, s);
}

}  // namespace ttt
