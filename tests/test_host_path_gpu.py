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


def layer_of(P, c, K):
    v = to_dev(c)
    H, d = v["W0"].shape[0], v["W0"].shape[1]
    layer = P.FusedTileMulti(P.ModelConfig(H, d, P.TTTConfig(mini_batch_size=K)), v["W0"], v["b0"], v["gamma"], v["beta"])
    return layer, P.TTTInputsInner(P.Qkv(v["xq"], v["xk"], v["xv"]), v["token_eta"], v["lr"])


@pytest.mark.parametrize("seq", [48, 39, 7])
def test_layer_takes_a_state_shared_over_the_batch(P, seq):
    """The layer's own parameters ([H,d,d], [H,d]) as a state give what their repetition over the batch gives: whole
    mini-batches, a remainder behind them, a remainder alone."""
    print(f"case layer, shared state, {seq} tokens", flush=True)
    B, H, d, K = 3, 2, 64, 16
    c = P.synthetic.reference_test_inputs(77, B, H, 48, d, K, io_dtype=torch.float32)
    for k in ("xq", "xk", "xv"):
        c[k] = c[k][:, :, :seq].contiguous()
    c["lr"] = c["lr"][:, :, :seq].contiguous()
    c["token_eta"] = c["token_eta"].repeat(48)[:seq].contiguous()
    layer, x = layer_of(P, c, K)
    for call in (lambda s: layer.forward(s, x), lambda s: layer.forward_mini_batch(s, x, range(0, min(seq, K)))):
        shared, full = P.TTTLinearState(layer.weight_init, layer.bias_init), layer.init_state(B)
        o1, o2 = call(shared), call(full)
        assert torch.equal(o1, o2) and torch.equal(shared.weight, full.weight) and torch.equal(shared.bias, full.bias)
        assert shared.weight.shape == (B, H, d, d)


def test_layer_needs_token_eta_of_a_mini_batch_only(P):
    """Whole mini-batches read the first K entries; a remainder reads those at its own tokens, and is refused without."""
    print("case layer, token_eta of K entries", flush=True)
    B, H, d, K = 2, 2, 64, 16
    c = P.synthetic.reference_test_inputs(78, B, H, 48, d, K, io_dtype=torch.float32)
    te = c["token_eta"][:K].contiguous()
    c["token_eta"] = te.repeat(3)
    layer, x = layer_of(P, c, K)
    short = P.TTTInputsInner(x.qkv, te.to("cuda:0"), x.ttt_lr_eta)
    s1, s2 = layer.init_state(B), layer.init_state(B)
    assert torch.equal(layer.forward(s1, short), layer.forward(s2, x)) and torch.equal(s1.weight, s2.weight)
    s1, s2 = layer.init_state(B), layer.init_state(B)
    r = range(0, K)
    assert torch.equal(layer.forward_mini_batch(s1, short, r), layer.forward_mini_batch(s2, x, r))
    cut = lambda t: t[:, :, :39].contiguous()
    short = P.TTTInputsInner(P.Qkv(cut(x.qkv.xq), cut(x.qkv.xk), cut(x.qkv.xv)), te.to("cuda:0"), cut(x.ttt_lr_eta))
    with pytest.raises(P.TttError, match="token_eta"):
        layer.forward(layer.init_state(B), short)


def test_layer_takes_a_sequence_without_tokens(P):
    print("case layer, empty sequence", flush=True)
    c = P.synthetic.reference_test_inputs(79, 2, 2, 16, 64, 16, io_dtype=torch.bfloat16)
    layer, x = layer_of(P, c, 16)
    cut = lambda t: t[:, :, :0]
    state = layer.init_state(2)
    W, b = state.weight, state.bias
    out = layer.forward(state, P.TTTInputsInner(P.Qkv(cut(x.qkv.xq), cut(x.qkv.xk), cut(x.qkv.xv)), x.token_eta[:0],
                                                cut(x.ttt_lr_eta)))
    assert out.shape == (2, 2, 0, 64) and out.dtype == torch.bfloat16
    assert state.weight is W and state.bias is b


def test_layer_refuses_a_mini_batch_without_tokens(P):
    print("case layer, mini_batch 0", flush=True)
    c = P.synthetic.reference_test_inputs(80, 1, 1, 16, 32, 16, io_dtype=torch.float32)
    layer, x = layer_of(P, c, 0)
    with pytest.raises(P.TttError, match="mini_batch 0"):
        layer.forward(layer.init_state(1), x)


def off_by_one(t):
    """The same contiguous tensor on the device, one element behind a 16-byte boundary."""
    return torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda:0")[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16], ids=["f32", "bf16"])
def test_sparse_linear_backward_takes_unaligned_tensors(P, dtype):
    """Coarser checkpoints than one per mini-batch: the kernel without a workspace reads element by element, so the call
    that is given one takes the same tensors (and workspaces)."""
    print(f"case sparse linear bwd, unaligned {dtype}", flush=True)
    B, H, d, K, N, ci = 2, 2, 64, 16, 5, 2
    c = P.synthetic.reference_test_inputs(81, B, H, N * K, d, K, io_dtype=dtype)
    dO = torch.randn(B, H, N * K, d, generator=torch.Generator().manual_seed(13)).to(dtype)
    v = to_dev(c)
    a = [v["xq"], v["xk"], v["xv"], v["W0"], v["b0"], v["token_eta"], v["lr"], v["gamma"], v["beta"]]
    Wc, bc = P.ttt_linear_forward_raw(*a, K, 1e-6, ci, want_checkpoints=True)[3:]
    ref = oracle_bwd(c, dO, K)
    got = P.ttt_linear_backward_raw(*[off_by_one(t) for t in a[:3]], *a[3:], Wc, bc, off_by_one(dO), K, 1e-6, ci)
    torch.cuda.synchronize()
    compare(got, ref, TOL[dtype])
    # a desc that needs no workspace ignores the one it is given
    ws = torch.empty(65, dtype=torch.uint8, device="cuda:0")[1:]
    got = P.ttt_linear_backward_raw(*a, Wc, bc, dO.to("cuda:0"), K, 1e-6, ci, kernel_hint=P.TTT_HINT_LDS_TILES, workspace=ws)
    torch.cuda.synchronize()
    compare(got, ref, TOL[dtype])
