"""GPU parity of ttt_linear_adam_fwd where the number of (batch, head) units chooses the kernel: past one unit per CU at
head_dim 64 and past two at head_dim 32, whole and short mini-batches, more mini-batches than the prefetch ring holds."""
import importlib

import numpy as np
import pytest
import torch

from helpers import TOL, np_inputs, to_dev
from oracle import ttt_oracle as orc
from test_linear_adam_gpu import HP, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("B,H,d,K,N", [(33, 8, 64, 16, 2), (33, 8, 64, 9, 2), (43, 12, 32, 16, 2), (1, 1, 64, 16, 7)])
def test_linear_adam_fwd_many_units(B, H, d, K, N, dtype):
    print(f"case linear adam B{B} H{H} d{d} K{K} N{N} {dtype}", flush=True)
    P = importlib.import_module("ttt-rs_amd")
    c = P.synthetic.reference_test_inputs(1700 + d + K + N, B, H, N * K, d, K, io_dtype=dtype)
    out, W, b, mo, _ = run(P, to_dev(c), K, **HP)
    n = np_inputs(c)
    ro, st = orc.linear_adam_forward(n["W0"], n["b0"], n["xq"], n["xk"], n["xv"], n["token_eta"], n["lr"], n["gamma"],
                                     n["beta"], K=K, **HP)
    for got, ref, name in zip((out, *mo), (ro, st["Wm"], st["bm"], st["Wv"], st["bv"]), ("out", "Wm", "bm", "Wv", "bv")):
        e = np.linalg.norm(got.double().cpu().numpy() - ref) / np.linalg.norm(ref)
        assert e <= TOL[dtype], f"{name}: relative error {e:.2e}"
    # an element whose gradient is nearly zero may move either way (the step has the size of the rate whatever the
    # gradient's), so the movement of the state is compared over nearly all elements
    for got, ref in ((W, st["W"]), (b, st["b"])):
        err = np.abs(got.double().cpu().numpy() - ref)
        assert (err <= 0.05 * HP["adam_lr"] * N).mean() >= (0.999 if dtype == torch.float32 else 0.95)
