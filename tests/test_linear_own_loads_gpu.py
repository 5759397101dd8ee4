"""GPU: the bf16 TTT-Linear forward whose waves load only the features they own: short mini-batches, one and two of them, and the
last buffer of the ring.  At head_dim 32 and 64 against the form in which every wave loads every row, bit for bit, what is saved
for a backward included (by the gradients that come of it: the buffers are larger than what is written).  At head_dim 96 and 128
it is the only form, and the hints select nothing: there the comparison shows that calls repeat, and the oracle the rest."""
import importlib

import pytest
import torch

from helpers import TOL, assert_close, to_dev
from test_linear_fwd_gpu import oracle_case
from test_repeat_calls_gpu import PLAIN_LINEAR

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    return importlib.import_module("ttt-rs_amd")


@pytest.mark.parametrize("fmt", [None, 0, 1, 2], ids=["no-ckpt", "f32-ckpt", "packed", "factors"])
@pytest.mark.parametrize("d,B,H,K,N", [
    (32, 1, 3, 16, 1), (32, 2, 2, 16, 5), (32, 1, 2, 7, 4), (64, 4, 8, 16, 9), (64, 3, 11, 16, 9), (64, 1, 2, 16, 8),
    (64, 1, 2, 5, 9), (96, 1, 2, 16, 1), (96, 2, 2, 16, 4), (96, 1, 2, 5, 7), (128, 1, 2, 16, 1), (128, 2, 2, 16, 2),
    (128, 1, 2, 3, 7), (128, 1, 1, 16, 5)])
def test_own_loads(P, d, B, H, K, N, fmt):
    if fmt == 2 and (d > 96 or N < 2):
        pytest.skip("update factors: head_dim <= 96, two or more mini-batches")
    print(f"case own loads d{d} B{B} H{H} K{K} N{N} fmt{fmt}", flush=True)
    c = P.synthetic.reference_test_inputs(4100 + d + K + N, B, H, N * K, d, K, io_dtype=torch.bfloat16)
    v = to_dev(c)
    dO = torch.randn(B, H, N * K, d, generator=torch.Generator().manual_seed(37)).to(torch.bfloat16).to("cuda:0")
    runs = []
    for hint in (0, P.TTT_HINT_ALL_LOADS, P.TTT_HINT_OWN_LOADS):
        r = P.ttt_linear_forward_raw(v["xq"], v["xk"], v["xv"], v["W0"], v["b0"], v["token_eta"], v["lr"], v["gamma"], v["beta"],
                                     K, 1e-6, 1, want_checkpoints=fmt is not None, packed_checkpoints=fmt or 0, kernel_hint=hint)
        runs.append(tuple(r) if fmt in (None, 0) else tuple(r[:3]))
        if fmt in (1, 2):
            g = P.ttt_linear_backward_raw(v["xq"], v["xk"], v["xv"], v["W0"], v["b0"], v["token_eta"], v["lr"], v["gamma"],
                                          v["beta"], r[3], r[4], dO, K, 1e-6, 1, packed_checkpoints=fmt)
            runs[-1] += tuple(g[k] for k in PLAIN_LINEAR)
        torch.cuda.synchronize()
    for r in runs[1:]:
        for i, (x, y) in enumerate(zip(runs[0], r)):
            assert torch.equal(x, y), f"output {i} depends on who loads the rows"
    for name, got, ref in zip(("out", "W", "b"), runs[0], oracle_case(c, K)):
        assert_close(got, ref, TOL[torch.bfloat16], name)
