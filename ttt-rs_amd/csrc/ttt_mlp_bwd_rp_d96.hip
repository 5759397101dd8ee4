// The register-resident TTT-MLP backward at head_dim 96: a translation unit of its own for a compiler option that the
// others do without (see build.py).
#include "ttt_mlp_bwd_rp.hip.h"

namespace ttt {

hipError_t launch_mlp_bwd_rp_d96(const MlpBwdRpArgs& a, hipStream_t s) { return launch_mlp_bwd_rp_d<96>(a, s); }

}  // namespace ttt
