"""ttt_mlpn_fwd with a unit on two workgroups: the same bits as on one (TTT_HINT_ONE_WORKGROUP), also where the partners do not
share an L2 (a release per mini-batch), where buffers that do not qualify keep a unit on one, and where the two wait for each
other in vain."""
import ctypes
import importlib

import pytest
import torch

from helpers import TOL, assert_close, np_inputs, to_dev
from oracle import ttt_oracle as orc
from test_mlpn_gpu import make_case

pytestmark = pytest.mark.gpu

ONE, LOST, OTHER_XCD = 0x8000, 0x200, 0x800


def call(P, c, Ws, bs, B, H, N, K, d, n_hidden, dtype, hint, skew=0, window=0, in_place=()):
    """Ws, bs: per head, or per batch element too.  window: tokens in front of and behind the N mini-batches in the buffers of the
    rows, which nothing may touch.  in_place: "W" (the first and the last weights over each other's initial ones), "b" (over the
    initial ones), "out" (over xq), "rows" (xq inside the second weights' output)."""
    seq, m, dev = N * K, 4 * d, "cuda:0"
    dims = [d] + [m] * n_hidden + [d]
    dv = to_dev(c)
    if window:
        for k in ("xq", "xk", "xv", "lr"):
            full = torch.full((B, H, seq + 2 * window, *dv[k].shape[3:]), float("nan"), dtype=dtype, device=dev)
            full[:, :, window:window + seq] = dv[k]
            dv[k] = full
    W0, b0 = [w.to(dev) for w in Ws], [b.to(dev) for b in bs]
    raw = [torch.full((B * H * dims[i] * dims[i + 1] + 4,), 7.0, device=dev) for i in range(n_hidden + 1)]
    Wo = [r[skew:skew + B * H * dims[i] * dims[i + 1]] for i, r in enumerate(raw)]
    bo = [torch.empty(B * H * dims[i + 1], device=dev) for i in range(n_hidden + 1)]
    out = dv["xq"] if "out" in in_place else torch.full_like(dv["xq"], 7.0)
    bo = b0 if "b" in in_place else bo
    if "W" in in_place:
        Wo[0], Wo[-1] = W0[-1].view(-1), W0[0].view(-1)
    if "rows" in in_place:
        into = Wo[1].view(dtype)[:dv["xq"].numel()].view_as(dv["xq"])
        dv["xq"] = into.copy_(dv["xq"])
    desc = P.TttDesc(B, H, seq, d, K, 1e-6, 1, P.TTT_BF16 if dtype == torch.bfloat16 else P.TTT_F32)
    desc.kernel_hint, desc.state_per_batch, desc.seq_stride = hint, int(Ws[0].dim() == 4), seq + 2 * window if window else 0
    arr = lambda ts: (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    row = lambda t: ctypes.c_void_p(t[0, 0, window].data_ptr())
    rc = P.lib().ttt_mlpn_fwd(ctypes.byref(desc), n_hidden, row(dv["xq"]), row(dv["xk"]), row(dv["xv"]), arr(W0), arr(b0),
                              p(dv["token_eta"]), row(dv["lr"]), p(dv["gamma"]), p(dv["beta"]), row(out), arr(Wo), arr(bo),
                              ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, P.lib().ttt_last_error()
    torch.cuda.synchronize()
    if window:
        edge = torch.cat([out[:, :, :window], out[:, :, window + seq:]], 2)
        assert (edge == 7.0).all(), "written outside the window"
        out = out[:, :, window:window + seq]
    return [out.contiguous(), *[w.reshape(-1) for w in Wo], *[b.reshape(-1) for b in bo]]


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


def per_batch(ts, B):
    """A state of its own for every batch element."""
    return [torch.stack([t * (1 + 0.25 * b) + 0.01 * b for b in range(B)]) for t in ts]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("n_hidden,B,H,d,K,N", [(2, 3, 2, 64, 16, 5), (3, 3, 3, 32, 7, 9)])
def test_carried_states_and_windows(n_hidden, B, H, d, K, N, dtype):
    """A state per batch element and a window of a longer sequence, with partners on one XCD, on two, and never together: the bits of
    one workgroup on packed rows."""
    print(f"case mlpn pair forms hidden{n_hidden} B{B} H{H} d{d} K{K} N{N} {dtype}", flush=True)
    P = importlib.import_module("ttt-rs_amd")
    c, Ws, bs = make_case(P, 2600 + n_hidden, B, H, N * K, d, K, n_hidden, dtype)
    shapes = (B, H, N, K, d, n_hidden, dtype)
    shared = call(P, c, Ws, bs, *shapes, ONE)
    Wp, bp = per_batch(Ws, B), per_batch(bs, B)
    own = call(P, c, Wp, bp, *shapes, ONE)
    assert not torch.equal(own[1], shared[1])
    for state, want in (((Ws, bs), shared), ((Wp, bp), own)):
        for kw in (dict(), dict(window=2 * K), dict(hint=OTHER_XCD, window=4 * K), dict(hint=LOST, window=K)):
            kw = dict(hint=0, **kw) if "hint" not in kw else kw
            for i, (a, b) in enumerate(zip(call(P, c, *state, *shapes, **kw), want)):
                assert torch.equal(a, b), (kw, i)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("n_hidden,B,H,d,K,N,over", [(3, 3, 3, 32, 7, 9, ("W",)), (2, 2, 2, 32, 16, 5, ("W", "b", "out")), (2, 2, 3, 64, 16, 5, ("out",)),
                                                     (2, 1, 1, 64, 16, 6, ("rows",)), (4, 1, 1, 32, 16, 6, ("rows", "b"))])
def test_outputs_over_inputs_keep_a_unit_on_one_workgroup(n_hidden, B, H, d, K, N, over, dtype):
    """What one workgroup has read before it writes, two would still read: the results are those with buffers of their own, and with
    the hint that makes partners give up nobody waited.  Biases alone may lie over the initial ones: each side reads those first."""
    print(f"case mlpn pair overlap hidden{n_hidden} B{B} H{H} d{d} K{K} N{N} {over} {dtype}", flush=True)
    P = importlib.import_module("ttt-rs_amd")
    c, Ws, bs = make_case(P, 2650 + n_hidden, B, H, N * K, d, K, n_hidden, dtype)
    shapes, state = (B, H, N, K, d, n_hidden, dtype), (per_batch(Ws, B), per_batch(bs, B))
    want, before = call(P, c, *state, *shapes, ONE), P.mlp_fwd_lost_workgroups()
    for hint in (LOST, 0):
        for i, (a, b) in enumerate(zip(call(P, c, *state, *shapes, hint, in_place=over), want)):
            assert torch.equal(a, b), (hint, i)
    assert P.mlp_fwd_lost_workgroups() == before
    for i, (a, b) in enumerate(zip(call(P, c, *state, *shapes, LOST, in_place=("b",)), want)):
        assert torch.equal(a, b), i
    assert P.mlp_fwd_lost_workgroups() == before + 2 * B * H


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
@pytest.mark.parametrize("n_hidden,B,H,d,K,N", [(2, 2, 1, 64, 16, 6), (3, 2, 2, 32, 16, 5), (4, 2, 1, 32, 5, 7)])
def test_two_workgroups_match_the_oracle(n_hidden, B, H, d, K, N, dtype):
    print(f"case mlpn pair oracle hidden{n_hidden} B{B} H{H} d{d} K{K} N{N} {dtype}", flush=True)
    P = importlib.import_module("ttt-rs_amd")
    c, Ws, bs = make_case(P, 2700 + n_hidden, B, H, N * K, d, K, n_hidden, dtype)
    n, f64 = np_inputs(c), lambda ts: [t.double().numpy() for t in ts]
    ro, rW, rb = orc.mlpn_forward(f64(Ws), f64(bs), n["xq"], n["xk"], n["xv"], n["token_eta"], n["lr"], n["gamma"], n["beta"], K=K)
    got = call(P, c, Ws, bs, B, H, N, K, d, n_hidden, dtype, 0)
    assert_close(got[0], ro, TOL[dtype], "out")
    for i in range(n_hidden + 1):  # f32 products for both I/O types: the bars of the one-workgroup test
        assert_close(got[1 + i].reshape(rW[i].shape), rW[i], 1e-4, f"W[{i}]")
        assert_close(got[2 + n_hidden + i].reshape(rb[i].shape), rb[i], 1e-4, f"b[{i}]", min_frac=0.99)


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
