"""What the host path between torch tensors and the C ABI (csrc/ttt_torch.cpp) takes and hands on, on the GPU."""
import importlib

import pytest
import torch

from helpers import TOL, to_dev
from test_linear_bwd_gpu import compare, oracle_bwd

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    return importlib.import_module("ttt-rs_amd")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("ci", [1, 3])
@pytest.mark.parametrize("given", ["weight", "bias"])
def test_linear_backward_takes_each_state_gradient_alone(P, given, ci, dtype):
    """d_W_out and d_b_out are optional one by one: the other counts as zero."""
    print(f"case linear bwd with grad_{given}_out only, ci{ci} {dtype}", flush=True)
    B, H, d, K, N = 2, 2, 64, 16, 4
    c = P.synthetic.reference_test_inputs(911 + ci, B, H, N * K, d, K, io_dtype=dtype)
    g = torch.Generator().manual_seed(12)
    dO = torch.randn(B, H, N * K, d, generator=g).to(dtype)
    sg = [torch.randn(B, H, d, d, generator=g), torch.randn(B, H, d, generator=g)]
    sg[1 if given == "weight" else 0].zero_()
    v = to_dev(c)
    a = (v["xq"], v["xk"], v["xv"], v["W0"], v["b0"], v["token_eta"], v["lr"], v["gamma"], v["beta"])
    Wc, bc = P.ttt_linear_forward_raw(*a, K, 1e-6, ci, want_checkpoints=True)[3:]
    kw = {f"grad_{given}_out": sg[0 if given == "weight" else 1].to("cuda:0")}
    got = P.ttt_linear_backward_raw(*a, Wc, bc, dO.to("cuda:0"), K, 1e-6, ci, **kw)
    torch.cuda.synchronize()
    compare(got, oracle_bwd(c, dO, K, sg), TOL[dtype])
