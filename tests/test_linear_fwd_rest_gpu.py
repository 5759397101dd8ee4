"""ttt_linear_fwd_with_rest: the whole mini-batches of a sequence and the short one behind them in one launch, against the two
launches it takes the place of: the same bits, also where the consumer waits in vain and the units are computed again, so that a
sequence's result does not depend on how many others are in its batch, on the language of the caller or on timing."""
import ctypes
import importlib

import pytest
import torch

from helpers import to_dev

pytestmark = pytest.mark.gpu

ONE, LOST, OTHER_XCD, HALFWAY = 0x8000, 0x200, 0x800, 0x10000
K = 16


@pytest.fixture(scope="module")
def P():
    return importlib.import_module("ttt-rs_amd")


def inputs(P, d, B, H, N, rest):
    seq = N * K + rest
    v = to_dev(P.synthetic.reference_test_inputs(5500 + d + N + rest, B, H, (N + 1) * K, d, K, io_dtype=torch.float32))
    for k in ("xq", "xk", "xv", "lr"):
        v[k] = v[k][:, :, :seq].contiguous()
    te = v["token_eta"]
    v["token_eta"] = torch.cat([te[:K].repeat(N), te[:rest] * 1.25]).contiguous()
    return v


def run(P, v, d, B, H, N, rest, hint, one_launch, shift=0):
    """shift: elements that the final weights lie off a 16-byte boundary."""
    seq, dev = N * K + rest, "cuda:0"
    buf = torch.full((B * H * seq * d + 16 * d,), 7.0, device=dev)  # behind the last row nothing may be written
    W = torch.full((2 * B * H * d * d + 4,), 7.0, device=dev)[shift:][:2 * B * H * d * d].view(2, B, H, d, d)
    b = torch.full((2, B, H, d), 7.0, device=dev)
    p = lambda t, at=0: ctypes.c_void_p(t.data_ptr() + 4 * at)
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)

    def desc(n, k, per_batch):
        ds = P.TttDesc(B, H, n, d, k, 1e-6, 1, P.TTT_F32)
        ds.kernel_hint, ds.seq_stride, ds.state_per_batch = hint, seq, per_batch
        return ctypes.byref(ds)

    def rows(at):
        return [p(v[k], at * d) for k in ("xq", "xk", "xv")]

    L, full = P.lib(), N * K
    if one_launch:
        rc = L.ttt_linear_fwd_with_rest(desc(full, K, 0), rest, *rows(0), p(v["W0"]), p(v["b0"]), p(v["token_eta"]), p(v["lr"]),
                                        p(v["gamma"]), p(v["beta"]), p(buf), p(W[1]), p(b[1]), s)
        assert rc == 0, L.ttt_last_error()
    else:
        for n, k, at, i in ((full, K, 0, 0), (rest, rest, full, 1)):
            state = (p(W[0]), p(b[0])) if i else (p(v["W0"]), p(v["b0"]))
            rc = L.ttt_linear_fwd(desc(n, k, i), *rows(at), *state, p(v["token_eta"], at), p(v["lr"], at), p(v["gamma"]),
                                  p(v["beta"]), p(buf, at * d), p(W[i]), p(b[i]), None, None, s)
            assert rc == 0, L.ttt_last_error()
    torch.cuda.synchronize()
    assert (buf[B * H * seq * d:] == 7.0).all(), "written behind the last row"
    return buf[:B * H * seq * d], W[1], b[1]


# one token, one short of a mini-batch; odd and even numbers of mini-batches; the fewest; units beyond a group of eight
@pytest.mark.parametrize("d,B,H,N,rest", [(64, 1, 1, 4, 1), (64, 3, 3, 5, 15), (64, 2, 12, 63, 5), (64, 8, 16, 8, 8), (32, 1, 2, 5, 1),
                                          (32, 3, 11, 16, 15), (32, 2, 4, 7, 7)])
@pytest.mark.parametrize("no_update", [False, True])
def test_equals_two_launches(P, d, B, H, N, rest, no_update):
    print(f"case linear rest d{d} B{B} H{H} N{N} rest{rest} {no_update}", flush=True)
    v = inputs(P, d, B, H, N, rest)
    if no_update:  # the short mini-batch leaves the state as it is
        v["token_eta"][-1] = 0.0
    two = run(P, v, d, B, H, N, rest, ONE, False)
    for hint in (0, OTHER_XCD, LOST, HALFWAY):
        for i, (x, y) in enumerate(zip(two, run(P, v, d, B, H, N, rest, hint, True))):
            assert torch.equal(x, y), f"output {i}, hint {hint:#x}"


@pytest.mark.parametrize("what", ["xq", "xk", "xv", "lr"])
@pytest.mark.parametrize("value", [float("inf"), float("nan"), 3e38])
def test_extremes_in_the_last_token(P, what, value):
    """The lanes behind the last token repeat nothing of it: the same values, infinities and NaN as two launches."""
    d, B, H, N, rest = 64, 1, 2, 5, 6
    print(f"case linear rest extremes {what} {value}", flush=True)
    v = inputs(P, d, B, H, N, rest)
    v[what][:, 0, -1] = value
    two = run(P, v, d, B, H, N, rest, ONE, False)
    for i, (x, y) in enumerate(zip(two, run(P, v, d, B, H, N, rest, 0, True))):
        assert torch.equal(x.isnan(), y.isnan()), f"output {i}"
        assert torch.equal(x.nan_to_num(0.0, 1.0, -1.0), y.nan_to_num(0.0, 1.0, -1.0)), f"output {i}"


# a batch whose units have two workgroups (f32) or a CU (bf16) to themselves, and the same sequences in one that has too many for that
@pytest.mark.parametrize("dtype,d,few,many", [(torch.float32, 64, 2, 12), (torch.float32, 32, 3, 11), (torch.bfloat16, 64, 4, 22)])
def test_bits_do_not_depend_on_the_batch(P, dtype, d, few, many):
    H, N, rest = 12, 5, 9
    seq = N * K + rest
    print(f"case linear rest batch {dtype} d{d}", flush=True)
    c = to_dev(P.synthetic.reference_test_inputs(5900 + d, many, H, seq, d, K, io_dtype=dtype))
    te = c["token_eta"].repeat(N + 1)[:seq].contiguous()
    layer = P.FusedTileMulti(P.ModelConfig(H, d, P.TTTConfig(mini_batch_size=K)), c["W0"], c["b0"], c["gamma"], c["beta"])

    def forward(B):
        st = layer.init_state(B)
        x = P.TTTInputsInner(P.Qkv(*(c[k][:B].contiguous() for k in ("xq", "xk", "xv"))), te, c["lr"][:B].contiguous())
        return layer.forward(st, x), st.weight, st.bias

    for i, (x, y) in enumerate(zip(forward(few), forward(many))):
        assert torch.equal(x, y[:few]), f"output {i}"


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_the_question_agrees_with_the_call(P, dtype):
    """ttt_linear_fwd_takes_rest against what ttt_linear_fwd_with_rest answers, around the limits in mini-batches, units and head_dim."""
    L, io, dev, rest = P.lib(), P.TTT_F32 if dtype == torch.float32 else P.TTT_BF16, "cuda:0", 3
    p = lambda t: ctypes.c_void_p(t.data_ptr())
    s = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    said = []
    for d in (32, 64, 96, 128):
        for B, H, N in ((1, 2, 3), (1, 2, 4), (8, 16, 4), (43, 3, 4), (16, 16, 4), (257, 1, 4), (32, 16, 4), (57, 9, 4)):
            seq = N * K + rest
            x, lr = torch.zeros(B, H, seq, d, device=dev, dtype=dtype), torch.zeros(B, H, seq, device=dev, dtype=dtype)
            out, te, one = torch.empty_like(x), torch.ones(seq, device=dev), torch.ones(H, d, d, device=dev)
            W, b = torch.empty(B, H, d, d, device=dev), torch.empty(B, H, d, device=dev)
            ds = P.TttDesc(B, H, N * K, d, K, 1e-6, 1, io)
            ds.seq_stride = seq
            print(f"case linear rest asked {dtype} d{d} B{B} H{H} N{N}", flush=True)
            asked = L.ttt_linear_fwd_takes_rest(ctypes.byref(ds), rest)
            rc = L.ttt_linear_fwd_with_rest(ctypes.byref(ds), rest, p(x), p(x), p(x), p(one), p(one), p(te), p(lr), p(one), p(one), p(out),
                                            p(W), p(b), s)
            torch.cuda.synchronize()
            assert rc == (P.TTT_OK if asked else P.TTT_ERR_UNSUPPORTED), (d, B, H, N)
            said.append(asked)
    assert 0 in said and 1 in said


def test_a_call_that_succeeds_leaves_no_error_text(P):
    """A layer's pass over a ragged sequence whose shape has no single launch."""
    v = inputs(P, 64, 1, 2, 3, 5)
    layer = P.FusedTileMulti(P.ModelConfig(2, 64, P.TTTConfig(mini_batch_size=K)), v["W0"], v["b0"], v["gamma"], v["beta"])
    print("case linear rest error text", flush=True)
    L = P.lib()
    assert L.ttt_linear_supported(None) == P.TTT_ERR_NULL
    before = L.ttt_last_error()
    layer.forward(layer.init_state(1), P.TTTInputsInner(P.Qkv(v["xq"], v["xk"], v["xv"]), v["token_eta"], v["lr"]))
    torch.cuda.synchronize()
    assert before and L.ttt_last_error() == before


def test_calls_without_one_launch_are_refused(P):
    v = inputs(P, 64, 1, 2, 3, 5)
    with pytest.raises(AssertionError, match="no single launch"):
        run(P, v, 64, 1, 2, 3, 5, 0, True)
    with pytest.raises(AssertionError, match="no single launch"):
        run(P, v, 64, 1, 2, 3, 5, ONE, True)


def test_final_weights_off_a_16_byte_boundary(P):
    """Two launches write them element by element; the one on two workgroups, where 16-byte accesses go there, does not take the call."""
    d, B, H, N, rest = 64, 1, 2, 5, 6
    v = inputs(P, d, B, H, N, rest)
    two = run(P, v, d, B, H, N, rest, 0, False)
    for shift in (1, 2, 3):
        print(f"case linear rest weights off by {shift}", flush=True)
        with pytest.raises(AssertionError, match="no single launch"):
            run(P, v, d, B, H, N, rest, 0, True, shift)
        for i, (x, y) in enumerate(zip(two, run(P, v, d, B, H, N, rest, 0, False, shift))):
            assert torch.equal(x, y), f"output {i}"


def test_layer_on_a_state_that_goes_on(P):
    """The layer's forward over a ragged sequence, twice, against its mini-batches one call each."""
    d, B, H, N, rest = 64, 2, 3, 6, 9
    v = inputs(P, d, B, H, N, rest)
    layer = P.FusedTileMulti(P.ModelConfig(H, d, P.TTTConfig(mini_batch_size=K)), v["W0"], v["b0"], v["gamma"], v["beta"])
    x = P.TTTInputsInner(P.Qkv(v["xq"], v["xk"], v["xv"]), v["token_eta"], v["lr"])
    seq = N * K + rest
    got, want = layer.init_state(B), layer.init_state(B)
    for _ in range(2):
        out = layer.forward(got, x)
        ref = torch.cat([layer.forward_mini_batch(want, x, range(i, min(i + K, seq))) for i in range(0, seq, K)], 2)
        for a, r in ((out, ref), (got.weight, want.weight), (got.bias, want.bias)):
            assert (a - r).abs().max() <= 1e-4 * r.abs().max()
