"""ttt_mlpn_fwd with a unit on two workgroups: the same bits as on one (TTT_HINT_ONE_WORKGROUP), also where the partners do not
share an L2 (a release per mini-batch), where buffers that do not qualify keep a unit on one, and where the two wait for each
other in vain."""
import ctypes
import importlib

import pytest
import torch

from helpers import to_dev
from test_mlpn_gpu import make_case

pytestmark = pytest.mark.gpu

ONE, LOST, OTHER_XCD = 0x8000, 0x200, 0x800


def call(P, c, Ws, bs, B, H, N, K, d, n_hidden, dtype, hint, skew=0):
    seq, m, dev = N * K, 4 * d, "cuda:0"
    dims = [d] + [m] * n_hidden + [d]
    dv = to_dev(c)
    W0, b0 = [w.to(dev) for w in Ws], [b.to(dev) for b in bs]
    raw = [torch.full((B * H * dims[i] * dims[i + 1] + 4,), 7.0, device=dev) for i in range(n_hidden + 1)]
    Wo = [r[skew:skew + B * H * dims[i] * dims[i + 1]] for i, r in enumerate(raw)]
    bo = [torch.empty(B * H * dims[i + 1], device=dev) for i in range(n_hidden + 1)]
    out = torch.empty_like(dv["xq"])
    desc = P.TttDesc(B, H, seq, d, K, 1e-6, 1, P.TTT_BF16 if dtype == torch.bfloat16 else P.TTT_F32)
    desc.kernel_hint = hint
    arr = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    rc = P.lib().ttt_mlpn_fwd(ctypes.byref(desc), n_hidden, p(dv["xq"]), p(dv["xk"]), p(dv["xv"]), arr(W0), arr(b0),
                              p(dv["token_eta"]), p(dv["lr"]), p(dv["gamma"]), p(dv["beta"]), p(out), arr(Wo), arr(bo),
                              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, P.lib().ttt_last_error()
    torch.cuda.synchronize()
    return [out, *Wo, *bo]


# the least number of mini-batches, one below it; a ring gone through several times; units beyond a group of eight, all CUs, more
CASES = [(2, 1, 1, 64, 16, 4), (2, 1, 1, 64, 16, 3), (2, 3, 3, 64, 16, 9), (2, 1, 5, 64, 7, 5), (2, 3, 3, 32, 16, 9),
         (3, 1, 9, 32, 16, 7), (4, 2, 4, 32, 1, 6), (4, 1, 3, 32, 16, 12), (2, 8, 16, 64, 16, 4), (2, 1, 129, 64, 16, 4)]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("n_hidden,B,H,d,K,N", CASES)
def test_two_workgroups_give_the_bits_of_one(n_hidden, B, H, d, K, N, dtype):
    print(f"case mlpn pair hidden{n_hidden} B{B} H{H} d{d} K{K} N{N} {dtype}", flush=True)
    P = importlib.import_module("ttt-rs_amd")
    c, Ws, bs = make_case(P, 2300 + n_hidden + d + K, B, H, N * K, d, K, n_hidden, dtype)
    args = (P, c, Ws, bs, B, H, N, K, d, n_hidden, dtype)
    one = call(*args, ONE)
    assert all(torch.isfinite(t).all() for t in one)
    for hint, skew in ((0, 0), (0, 0), (OTHER_XCD, 0), (0, 1)):
        for a, b in zip(call(*args, hint, skew), one):
            assert torch.equal(a, b), (hint, skew)


@pytest.mark.parametrize("n_hidden,B,H,d,K,N", [(2, 1, 2, 64, 16, 9), (3, 1, 9, 32, 5, 9), (2, 1, 128, 32, 16, 9)])
def test_units_that_wait_in_vain_are_done_again(n_hidden, B, H, d, K, N):
    """No workgroup finds its partner (they give up at once): the counter says so, the results are those of one workgroup."""
    P = importlib.import_module("ttt-rs_amd")
    c, Ws, bs = make_case(P, 2400, B, H, N * K, d, K, n_hidden, torch.float32)
    args = (P, c, Ws, bs, B, H, N, K, d, n_hidden, torch.float32)
    one, before = call(*args, ONE), P.mlp_fwd_lost_workgroups()
    got = call(*args, LOST)
    assert P.mlp_fwd_lost_workgroups() == before + 2 * B * H
    for i, (a, b) in enumerate(zip(got, one)):
        assert torch.equal(a, b), i


def test_one_workgroup_can_be_asked_for_from_python():
    """kernel_hint reaches the library from the call and from the layer object: no workgroup waits where one was asked for."""
    P = importlib.import_module("ttt-rs_amd")
    B, H, d, K, N = 1, 2, 32, 16, 5
    c, Ws, bs = make_case(P, 2450, B, H, N * K, d, K, 2, torch.float32)
    dv, dev = to_dev(c), lambda ts: [t.to("cuda:0") for t in ts]
    x = (dv["xq"], dv["xk"], dv["xv"])
    before = P.mlp_fwd_lost_workgroups()

    def raw(hint):
        out, W, b = P.ttt_mlpn_forward_raw(*x, dev(Ws), dev(bs), dv["token_eta"], dv["lr"], dv["gamma"], dv["beta"], K, kernel_hint=hint)
        return [out, *W, *b]

    def layer(hint):
        m = P.FusedMlpN(P.ModelConfig(H, d, P.TTTConfig(mini_batch_size=K)), dev(Ws), dev(bs), dv["gamma"], dv["beta"], kernel_hint=hint)
        state = m.init_state(B)
        out = m.forward(state, P.TTTInputsInner(P.Qkv(*x), dv["token_eta"].repeat(N), dv["lr"]))
        return [out, *state.weights, *state.biases]

    want = raw(ONE | LOST)
    for f in (raw, layer):
        for a, b in zip(f(ONE | LOST), want):
            assert torch.equal(a, b)
    assert P.mlp_fwd_lost_workgroups() == before
    for i, f in enumerate((raw, layer)):
        for a, b in zip(f(LOST), want):
            assert torch.equal(a, b)
        assert P.mlp_fwd_lost_workgroups() == before + 2 * B * H * (i + 1)


def test_two_workgroups_in_a_graph():
    P = importlib.import_module("ttt-rs_amd")
    B, H, d, K, N = 2, 3, 64, 16, 5
    c, Ws, bs = make_case(P, 2500, B, H, N * K, d, K, 2, torch.bfloat16)
    dv, dev = to_dev(c), lambda ts: [t.to("cuda:0") for t in ts]
    W0, b0 = dev(Ws), dev(bs)
    run = lambda: P.ttt_mlpn_forward_raw(dv["xq"], dv["xk"], dv["xv"], W0, b0, dv["token_eta"], dv["lr"], dv["gamma"], dv["beta"], K)
    want = run()
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        run()
    torch.cuda.current_stream().wait_stream(s)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for _ in range(3):
        for t in (got[0], *got[1], *got[2]):
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for a, b in zip((got[0], *got[1], *got[2]), (want[0], *want[1], *want[2])):
            assert torch.equal(a, b)
