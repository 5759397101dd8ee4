"""GPU parity of the register-resident TTT-MLP backward (bf16 I/O, head_dim 32 / 64 / 96) where its own structure can go
wrong: sequences longer than its hand-over slots, on two workgroups per unit (a ring) and on one (a launch per slots)."""
import importlib

import pytest
import torch

from helpers import TOL, assert_close
from test_mlp_bwd_gpu import GRADS, run_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    return importlib.import_module("ttt-rs_amd")


@pytest.mark.parametrize("B,H,d,K,N,sg", [(1, 2, 32, 16, 2, True), (1, 1, 64, 16, 4, False), (1, 2, 96, 11, 19, True),
                                          (1, 1, 96, 16, 64, False), (2, 5, 64, 16, 33, True)])
def test_register_resident_backward(P, B, H, d, K, N, sg):
    print(f"case mlp bwd rp B{B} H{H} d{d} K{K} N{N} sg={sg}", flush=True)
    got, ref = run_case(P, B, H, d, K, N, torch.bfloat16, "baseline", sg)
    one, _ = run_case(P, B, H, d, K, N, torch.bfloat16, "baseline", sg, kernel_hint=P.TTT_HINT_ONE_WORKGROUP)
    for k in GRADS:
        # d_token_eta is a sum over units with alternating signs: few mini-batches leave little but rounding
        assert_close(got[k], ref[k], TOL[torch.bfloat16] * (5 if k == "d_token_eta" else 1), k, min_frac=0.8)
        if k in ("d_token_eta", "d_gamma", "d_beta"):  # atomic additions: their order is not fixed
            assert_close(one[k], got[k].double(), 1e-5, k)
        else:
            assert torch.equal(one[k], got[k]), f"{k}: one workgroup per unit differs from two"
