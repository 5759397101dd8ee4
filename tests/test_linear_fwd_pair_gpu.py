"""ttt_linear_fwd, f32 I/O, with a unit on two workgroups: the same bits as on one (TTT_HINT_ONE_WORKGROUP), output, final state and
checkpoints, also where the two do not share an L2 (a release per mini-batch), where buffers that do not qualify keep a unit
on one, and where the consumer waits in vain, from the start or half way, and the unit is computed again."""
import ctypes
import importlib

import pytest
import torch

from helpers import TOL, assert_close, to_dev
from test_linear_fwd_gpu import oracle_case

pytestmark = pytest.mark.gpu

ONE, LOST, OTHER_XCD, HALFWAY = 0x8000, 0x200, 0x800, 0x10000
K = 16


@pytest.fixture(scope="module")
def P():
    return importlib.import_module("ttt-rs_amd")


def make(P, d, B, H, N, seed, no_update=False):
    c = P.synthetic.reference_test_inputs(seed, B, H, N * K, d, K, io_dtype=torch.float32)
    if no_update:
        c["token_eta"] = c["token_eta"].clone()
        c["token_eta"][K - 1] = 0.0
    return c


def call(P, c, d, B, H, N, hint, ckpt=None, ci=1, window=0, in_place=()):
    """ckpt: None, 0 (f32 matrices) or 1 (packed).  window: tokens in front of and behind the N mini-batches in the buffers of
    the rows, which nothing may touch.  in_place: "W" (the final weights over the initial ones, per batch element), "out" (over xq)."""
    seq, dev = N * K, "cuda:0"
    v = to_dev(c)
    if window:
        for k in ("xq", "xk", "xv", "lr"):
            full = torch.full((B, H, seq + 2 * window, *v[k].shape[3:]), float("nan"), device=dev)
            full[:, :, window:window + seq] = v[k]
            v[k] = full
    out = v["xq"] if "out" in in_place else torch.full_like(v["xq"], 7.0)
    W0, b0 = v["W0"], v["b0"]
    if "W" in in_place:
        W0, b0 = (t.expand(B, *t.shape[-t.dim():]).contiguous() if t.dim() == n else t.contiguous() for t, n in ((W0, 3), (b0, 2)))
    W = W0 if "W" in in_place else torch.full((B, H, d, d), 7.0, device=dev)
    b = torch.full((B, H, d), 7.0, device=dev)
    desc = P.TttDesc(B, H, seq, d, K, 1e-6, ci, P.TTT_F32)
    desc.kernel_hint, desc.state_per_batch, desc.seq_stride = hint, int(W0.dim() == 4), seq + 2 * window if window else 0
    desc.checkpoint_format = ckpt or 0
    n = -(-N // ci)
    Wc, bc = (torch.full(s, 7.0, device=dev) for s in ((B, H, n, d, d), (B, H, n, d)))
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    row = lambda t: ctypes.c_void_p(t[0, 0, window].data_ptr())
    rc = P.lib().ttt_linear_fwd(ctypes.byref(desc), row(v["xq"]), row(v["xk"]), row(v["xv"]), p(W0), p(b0), p(v["token_eta"]),
                                row(v["lr"]), p(v["gamma"]), p(v["beta"]), row(out), p(W), p(b),
                                p(Wc) if ckpt is not None else None, p(bc) if ckpt is not None else None,
                                ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    assert rc == 0, P.lib().ttt_last_error()
    torch.cuda.synchronize()
    if window:
        edge = torch.cat([out[:, :, :window], out[:, :, window + seq:]], 2)
        assert (edge == 7.0).all(), "written outside the window"
        out = out[:, :, window:window + seq].contiguous()
    return out, W, b, Wc, bc


# the least number of mini-batches and one below it; odd and even ones; units beyond a group of eight, half the CUs, more
CASES = [(64, 1, 1, 16), (64, 1, 1, 15), (64, 3, 3, 21), (64, 2, 12, 63), (64, 8, 16, 16), (64, 9, 15, 17), (32, 1, 2, 17),
         (32, 3, 11, 20), (32, 8, 16, 33)]


@pytest.mark.parametrize("d,B,H,N", CASES)
def test_same_bits_as_on_one_workgroup(P, d, B, H, N):
    print(f"case linear pair d{d} B{B} H{H} N{N}", flush=True)
    c = make(P, d, B, H, N, 5100 + d + N)
    one = call(P, c, d, B, H, N, ONE)
    for hint in (0, OTHER_XCD, LOST, HALFWAY):
        for i, (x, y) in enumerate(zip(one, call(P, c, d, B, H, N, hint))):
            assert torch.equal(x, y), f"output {i}, hint {hint:#x}"
    for name, got, ref in zip(("out", "W", "b"), one, oracle_case(c, K)):
        assert_close(got, ref, TOL[torch.float32], name)


@pytest.mark.parametrize("ckpt,ci", [(0, 1), (0, 3), (0, 16), (1, 1)])
@pytest.mark.parametrize("d,B,H,N", [(64, 2, 5, 17), (32, 2, 5, 17)])
def test_checkpoints(P, d, B, H, N, ckpt, ci):
    print(f"case linear pair checkpoints d{d} N{N} fmt{ckpt} ci{ci}", flush=True)
    c = make(P, d, B, H, N, 5200 + d)
    one = call(P, c, d, B, H, N, ONE, ckpt, ci)
    for hint in (0, LOST, HALFWAY):
        for i, (x, y) in enumerate(zip(one, call(P, c, d, B, H, N, hint, ckpt, ci))):
            assert torch.equal(x, y), f"output {i}, hint {hint:#x}"


@pytest.mark.parametrize("what", ["window", "no update", "W in place", "out in place"])
def test_other_calls(P, what):
    d, B, H, N = 64, 2, 3, 18
    print(f"case linear pair {what}", flush=True)
    c = make(P, d, B, H, N, 5300, no_update=what == "no update")
    kw = {"window": 16} if what == "window" else {"in_place": (what.split()[0],)} if "in place" in what else {}
    one = call(P, c, d, B, H, N, ONE, **kw)
    for hint in (0, OTHER_XCD, LOST, HALFWAY):
        for i, (x, y) in enumerate(zip(one, call(P, c, d, B, H, N, hint, **kw))):
            assert torch.equal(x, y), f"output {i}, hint {hint:#x}"
    if what == "no update":
        assert torch.equal(one[1][0], to_dev(c)["W0"])


def test_two_streams_and_replays(P):
    """Two calls at once, more workgroups than CUs; and a captured call, replayed between eager ones."""
    d, B, H, N = 64, 8, 12, 32
    print("case linear pair streams, graph", flush=True)
    c = make(P, d, B, H, N, 5400)
    v = to_dev(c)
    args = (v["xq"], v["xk"], v["xv"], v["W0"], v["b0"], v["token_eta"], v["lr"], v["gamma"], v["beta"], K)
    want = P.ttt_linear_forward_raw(*args, kernel_hint=ONE)
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
