"""ttt_linear_fwd, bf16 I/O, with the waves of a unit in roles (up to two units per CU): the same bits as the two-wave kernel
(TTT_HINT with two waves), output, final state, states and update factors; windows of a longer sequence; overlapping buffers."""
import ctypes
import importlib

import pytest
import torch

from helpers import TOL, assert_close, to_dev
from test_linear_fwd_gpu import oracle_case

pytestmark = pytest.mark.gpu

TWO_WAVES = 2
K = 16


@pytest.fixture(scope="module")
def P():
    return importlib.import_module("ttt-rs_amd")


def call(P, v, d, B, H, N, hint, ckpt=None, ci=1, window=0, in_place=False):
    seq, dev = N * K, "cuda:0"
    v = dict(v)
    if window:
        for k in ("xq", "xk", "xv", "lr"):
            full = torch.full((B, H, seq + 2 * window, *v[k].shape[3:]), float("nan"), device=dev, dtype=torch.bfloat16)
            full[:, :, window:window + seq] = v[k]
            v[k] = full
    out = v["xq"].clone() if in_place else torch.full_like(v["xq"], 7.0)
    xq = out if in_place else v["xq"]
    W, b = torch.full((B, H, d, d), 7.0, device=dev), torch.full((B, H, d), 7.0, device=dev)
    n = -(-N // ci)
    Wc, bc = torch.full((B, H, n, d, d), 7.0, device=dev), torch.full((B, H, n, d), 7.0, device=dev)
    desc = P.TttDesc(B, H, seq, d, K, 1e-6, ci, P.TTT_BF16)
    desc.kernel_hint, desc.seq_stride, desc.checkpoint_format = hint, seq + 2 * window if window else 0, ckpt or 0
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    row = lambda t: ctypes.c_void_p(t[0, 0, window].data_ptr())
    save = ckpt is not None
    rc = P.lib().ttt_linear_fwd(ctypes.byref(desc), row(xq), row(v["xk"]), row(v["xv"]), p(v["W0"]), p(v["b0"]), p(v["token_eta"]),
                                row(v["lr"]), p(v["gamma"]), p(v["beta"]), row(out), p(W), p(b), p(Wc) if save else None,
                                p(bc) if save else None, ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, P.lib().ttt_last_error()
    torch.cuda.synchronize()
    if window:
        edge = torch.cat([out[:, :, :window], out[:, :, window + seq:]], 2)
        assert (edge == 7.0).all(), "written outside the window"
        out = out[:, :, window:window + seq].contiguous()
    return out, W, b, Wc, bc


def make(P, d, B, H, N, no_update=False):
    c = P.synthetic.reference_test_inputs(5600 + d + N, B, H, N * K, d, K, io_dtype=torch.bfloat16)
    if no_update:
        c["token_eta"] = c["token_eta"].clone()
        c["token_eta"][K - 1] = 0.0
    return c


# one mini-batch, around the ring of eight, odd and even; a unit per CU, more (an odd number too), two per CU (head_dim 32; at 64 these
# are the two-wave kernel's)
@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("B,H,N", [(1, 1, 1), (1, 2, 2), (1, 3, 3), (2, 3, 7), (2, 3, 8), (3, 3, 9), (2, 5, 18), (16, 16, 5), (17, 16, 4),
                                   (24, 16, 11), (32, 16, 3), (257, 1, 3)])
def test_same_bits_as_two_waves(P, d, B, H, N):
    print(f"case linear roles d{d} B{B} H{H} N{N}", flush=True)
    c = make(P, d, B, H, N)
    v = to_dev(c)
    two, got = call(P, v, d, B, H, N, TWO_WAVES), call(P, v, d, B, H, N, 0)
    for i, (x, y) in enumerate(zip(two, got)):
        assert torch.equal(x, y), f"output {i}"
    if B * H < 16:
        for name, x, ref in zip(("out", "W", "b"), got, oracle_case(c, K)):
            assert_close(x, ref, TOL[torch.bfloat16], name)


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("ckpt,ci", [(0, 1), (0, 3), (1, 1), (2, 1)])
@pytest.mark.parametrize("B,H,N", [(2, 3, 10), (18, 16, 3), (1, 3, 1), (2, 3, 2), (3, 3, 3), (257, 1, 10), (32, 16, 9), (16, 16, 7)])
def test_saved(P, d, B, H, N, ckpt, ci):
    print(f"case linear roles saved d{d} B{B} H{H} N{N} fmt{ckpt} ci{ci}", flush=True)
    v = to_dev(make(P, d, B, H, N))
    for i, (x, y) in enumerate(zip(call(P, v, d, B, H, N, TWO_WAVES, ckpt, ci), call(P, v, d, B, H, N, 0, ckpt, ci))):
        assert torch.equal(x, y), f"output {i}"


@pytest.mark.parametrize("what", ["window", "no update", "out in place"])
@pytest.mark.parametrize("d,B,H,N", [(64, 2, 3, 13), (32, 20, 16, 6)])
def test_other_calls(P, d, B, H, N, what):
    print(f"case linear roles {what}", flush=True)
    v = to_dev(make(P, d, B, H, N, no_update=what == "no update"))
    kw = {"window": 32} if what == "window" else {"in_place": True} if what == "out in place" else {}
    two, got = call(P, v, d, B, H, N, TWO_WAVES, **kw), call(P, v, d, B, H, N, 0, **kw)
    for i, (x, y) in enumerate(zip(two, got)):
        assert torch.equal(x, y), f"output {i}"


# the fewest mini-batches, odd and even; one token and one short of a mini-batch; more than a unit per CU (head_dim 32)
@pytest.mark.parametrize("d,B,H,N,rest", [(64, 1, 1, 4, 1), (64, 2, 3, 5, 15), (64, 16, 16, 9, 6), (32, 2, 3, 4, 15), (32, 18, 16, 7, 1)])
@pytest.mark.parametrize("no_update", [False, True])
def test_rest_equals_two_launches(P, d, B, H, N, rest, no_update):
    """ttt_linear_fwd_with_rest against two launches: the same bits."""
    print(f"case linear roles rest d{d} B{B} H{H} N{N} rest{rest} {no_update}", flush=True)
    seq, full, dev = N * K + rest, N * K, "cuda:0"
    v = to_dev(P.synthetic.reference_test_inputs(5700 + d + N, B, H, (N + 1) * K, d, K, io_dtype=torch.bfloat16))
    for k in ("xq", "xk", "xv", "lr"):
        v[k] = v[k][:, :, :seq].contiguous()
    te = torch.cat([v["token_eta"][:K].repeat(N), v["token_eta"][:rest] * 1.25]).contiguous()
    if no_update:
        te[-1] = 0.0
    p = lambda t, at=0: ctypes.c_void_p(t.data_ptr() + t.element_size() * at)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    bufs = [torch.full((B * H * seq * d + 16 * d,), 7.0, device=dev, dtype=torch.bfloat16) for _ in range(2)]
    W, b = torch.full((3, B, H, d, d), 7.0, device=dev), torch.full((3, B, H, d), 7.0, device=dev)

    def desc(n, k, per_batch, hint):
        ds = P.TttDesc(B, H, n, d, k, 1e-6, 1, P.TTT_BF16)
        ds.kernel_hint, ds.seq_stride, ds.state_per_batch = hint, seq, per_batch
        return ctypes.byref(ds)

    rows = lambda at: [p(v[k], at * d) for k in ("xq", "xk", "xv")]
    for n, k, at, i in ((full, K, 0, 0), (rest, rest, full, 1)):
        state = (p(W[0]), p(b[0])) if i else (p(v["W0"]), p(v["b0"]))
        assert P.lib().ttt_linear_fwd(desc(n, k, i, TWO_WAVES), *rows(at), *state, p(te, at), p(v["lr"], at), p(v["gamma"]), p(v["beta"]),
                                      p(bufs[0], at * d), p(W[i]), p(b[i]), None, None, s) == 0
    assert P.lib().ttt_linear_fwd_with_rest(desc(full, K, 0, 0), rest, *rows(0), p(v["W0"]), p(v["b0"]), p(te), p(v["lr"]),
                                            p(v["gamma"]), p(v["beta"]), p(bufs[1]), p(W[2]), p(b[2]), s) == 0, P.lib().ttt_last_error()
    torch.cuda.synchronize()
    assert (bufs[1][B * H * seq * d:] == 7.0).all(), "written behind the last row"
    for name, x, y in (("out", *bufs), ("W", W[1], W[2]), ("b", b[1], b[2])):
        assert torch.equal(x, y), name


# one mini-batch, around the ring of eight; more than a unit per CU (head_dim 32)
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("d,B,H,N", [(64, 1, 3, 1), (64, 2, 5, 2), (64, 2, 3, 9), (64, 1, 12, 20), (64, 24, 16, 9), (32, 2, 3, 4), (32, 1, 5, 7), (32, 20, 16, 10),
                                     (32, 1, 3, 1), (32, 2, 3, 2), (32, 257, 1, 3)])
def test_operands_formed_from_projections(P, d, B, H, N, rope):
    """The fused call without copies of the operands against forming them first: the same bits."""
    print(f"case linear roles formed d{d} B{B} H{H} N{N} rope{rope}", flush=True)
    dev, seq = "cuda:0", N * K
    g = torch.Generator(device=dev).manual_seed(5800 + d + N)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)
    x = [r(B, seq, H, d).bfloat16() for _ in range(3)]
    args = (*x, r(B, seq, H).bfloat16(), r(H) * 0.5, 0.8, 1.0 / torch.arange(1, K + 1, dtype=torch.float32, device=dev), r(K) * 0.1)
    state = (r(H, d, d) * 0.02, r(H, d) * 0.02, 1.0 + 0.1 * r(H, d), 0.1 * r(H, d))
    _same_formed(P, args, state, dict(rope=P.rope_cos_sin(K, 0, None, d, dev), pos_offset=5, pos_wrap=K) if rope else {})


def _same_formed(P, args, state, pos):
    got = P.ttt_linear_forward_fused_inputs_raw(*args, *state, K, **pos)
    ins = P.inner_loop_inputs_raw(*args, K, **pos)
    want = P.ttt_linear_forward_raw(ins.qkv.xq, ins.qkv.xk, ins.qkv.xv, state[0], state[1], ins.token_eta, ins.ttt_lr_eta, *state[2:], K,
                                    kernel_hint=TWO_WAVES)
    torch.cuda.synchronize()
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), f"output {i}"


@pytest.mark.parametrize("wrap", [1, 2, 8])
def test_operands_formed_with_positions_that_repeat_within_the_mini_batch(P, wrap):
    d, B, H, N = 64, 1, 3, 3
    print(f"case linear roles formed wrap {wrap}", flush=True)
    dev, seq = "cuda:0", N * K
    g = torch.Generator(device=dev).manual_seed(5900 + wrap)
    r = lambda *s: torch.randn(*s, generator=g, device=dev)
    x = [r(B, seq, H, d).bfloat16() for _ in range(3)]
    args = (*x, r(B, seq, H).bfloat16(), r(H) * 0.5, 0.8, 1.0 / torch.arange(1, K + 1, dtype=torch.float32, device=dev), r(K) * 0.1)
    state = (r(H, d, d) * 0.02, r(H, d) * 0.02, 1.0 + 0.1 * r(H, d), 0.1 * r(H, d))
    _same_formed(P, args, state, dict(rope=P.rope_cos_sin(K, 0, None, d, dev), pos_offset=3, pos_wrap=wrap))


@pytest.mark.parametrize("in_place", [False, True])
@pytest.mark.parametrize("d,B,H", [(64, 2, 3), (32, 2, 3), (32, 20, 16)])
def test_a_state_per_batch_element_carried_through_windows(P, d, B, H, in_place):
    """Windows of 1, 3, 2 and 5 mini-batches of one sequence, each on the state the one before left, also over it in place."""
    print(f"case linear roles carried d{d} B{B} {in_place}", flush=True)
    N = 11
    v = to_dev(make(P, d, B, H, N))
    p = lambda t, at=0: ctypes.c_void_p(t.data_ptr() + t.element_size() * at)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    res = []
    for hint in (TWO_WAVES, 0):
        out = torch.full_like(v["xq"], 7.0)
        W, b = v["W0"].expand(B, H, d, d).contiguous(), v["b0"].expand(B, H, d).contiguous()
        at = 0
        for n in (1, 3, 2, 5):
            desc = P.TttDesc(B, H, n * K, d, K, 1e-6, 1, P.TTT_BF16)
            desc.kernel_hint, desc.seq_stride, desc.state_per_batch = hint, N * K, 1
            Wn, bn = (W, b) if in_place else (torch.empty_like(W), torch.empty_like(b))
            rc = P.lib().ttt_linear_fwd(ctypes.byref(desc), *[p(v[k], at * d) for k in ("xq", "xk", "xv")], p(W), p(b), p(v["token_eta"]),
                                        p(v["lr"], at), p(v["gamma"]), p(v["beta"]), p(out, at * d), p(Wn), p(bn), None, None, s)
            assert rc == 0, P.lib().ttt_last_error()
            W, b, at = Wn, bn, at + n * K
        torch.cuda.synchronize()
        res.append((out, W, b))
    for i, (x, y) in enumerate(zip(*res)):
        assert torch.equal(x, y), f"output {i}"


@pytest.mark.parametrize("what", ["xq", "xk", "xv", "lr"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3e38])
def test_extremes(P, what, value):
    """In the last token of a mini-batch and, for a sequence that ends in a short one, in its last token."""
    d, B, H, N, rest = 64, 1, 2, 5, 6
    print(f"case linear roles extremes {what} {value}", flush=True)
    v = to_dev(make(P, d, B, H, N))
    v[what][:, 0, 2 * K - 1] = value
    same = lambda x, y: torch.equal(x.isnan(), y.isnan()) and torch.equal(x.nan_to_num(0.0, 1.0, -1.0), y.nan_to_num(0.0, 1.0, -1.0))
    for i, (x, y) in enumerate(zip(call(P, v, d, B, H, N, TWO_WAVES), call(P, v, d, B, H, N, 0))):
        assert same(x.float(), y.float()), f"output {i}"
    c = to_dev(P.synthetic.reference_test_inputs(5950, B, H, N * K + rest, d, K, io_dtype=torch.bfloat16))
    c[what][:, 0, -1] = value
    te = c["token_eta"].repeat(N + 1)[:N * K + rest].contiguous()
    layer = P.FusedTileMulti(P.ModelConfig(H, d, P.TTTConfig(mini_batch_size=K)), c["W0"], c["b0"], c["gamma"], c["beta"])
    x = P.TTTInputsInner(P.Qkv(c["xq"], c["xk"], c["xv"]), te, c["lr"])
    one, two = layer.init_state(B), layer.init_state(B)
    a = layer.forward(one, x)
    whole = layer._pass(two, x, 0, N * K)
    b = torch.cat([whole, layer.forward_mini_batch(two, x, range(N * K, N * K + rest))], 2)
    for i, (p, q) in enumerate(((a, b), (one.weight, two.weight), (one.bias, two.bias))):
        assert same(p.float(), q.float()), f"ragged, output {i}"


def test_two_streams_and_replays(P):
    """Calls at once that do not fit side by side; a captured call, replayed between eager ones."""
    d, B, H, N = 64, 12, 16, 6
    print("case linear roles streams, graph", flush=True)
    v = to_dev(make(P, d, B, H, N))
    args = (v["xq"], v["xk"], v["xv"], v["W0"], v["b0"], v["token_eta"], v["lr"], v["gamma"], v["beta"], K)
    want = P.ttt_linear_forward_raw(*args, kernel_hint=TWO_WAVES)
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    got = []
    for s in streams * 3:
        with torch.cuda.stream(s):
            got.append(P.ttt_linear_forward_raw(*args))
    torch.cuda.synchronize()
    for r in got:
        for x, y in zip(r, want):
            assert torch.equal(x, y)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        res = P.ttt_linear_forward_raw(*args)
    for _ in range(3):
        for t in res:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        eager = P.ttt_linear_forward_raw(*args)
        torch.cuda.synchronize()
        for x, y, z in zip(res, want, eager):
            assert torch.equal(x, y) and torch.equal(z, y)
