"""ttt_mlpn_fwd against the float64 oracle where its tiles can go wrong: one token to a mini-batch, a mini-batch one short
of a tile, every depth, units beyond one XCD, and enough mini-batches that a state kept or fetched wrongly shows."""
import importlib

import pytest
import torch

from helpers import TOL, assert_close, np_inputs, to_dev
from oracle import ttt_oracle as orc
from test_mlpn_gpu import make_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("n_hidden,B,H,d,K,N", [(2, 1, 3, 64, 1, 5), (2, 3, 3, 64, 15, 9), (2, 1, 1, 64, 16, 24),
                                                (2, 1, 3, 32, 15, 9), (3, 3, 3, 32, 16, 17), (4, 1, 2, 32, 1, 5),
                                                (4, 2, 2, 32, 7, 12)])
def test_state_over_many_mini_batches(n_hidden, B, H, d, K, N, dtype):
    print(f"case mlpn hidden{n_hidden} B{B} H{H} d{d} K{K} N{N} {dtype}", flush=True)
    P = importlib.import_module("ttt-rs_amd")
    c, Ws, bs = make_case(P, 2100 + n_hidden + d + K, B, H, N * K, d, K, n_hidden, dtype)
    dv = to_dev(c)
    dev = lambda ts: [t.to("cuda:0") for t in ts]
    out, Wo, bo = P.ttt_mlpn_forward_raw(dv["xq"], dv["xk"], dv["xv"], dev(Ws), dev(bs), dv["token_eta"], dv["lr"],
                                         dv["gamma"], dv["beta"], K)
    torch.cuda.synchronize()
    n = np_inputs(c)
    ro, rW, rb = orc.mlpn_forward([w.double().numpy() for w in Ws], [b.double().numpy() for b in bs], n["xq"], n["xk"],
                                  n["xv"], n["token_eta"], n["lr"], n["gamma"], n["beta"], K=K)
    # f32 products for both I/O types: the state is held to 1e-4, the output to the I/O type's bar
    assert_close(out, ro, TOL[dtype], "out")
    for i in range(n_hidden + 1):
        assert_close(Wo[i], rW[i], 1e-4, f"W[{i}]")
        assert_close(bo[i], rb[i], 1e-4, f"b[{i}]", min_frac=0.99)
