"""GPU parity of the register-resident TTT-MLP backward (bf16 I/O, head_dim 32 / 64 / 96) where its own structure can go
wrong: sequences longer than its hand-over slots, on two workgroups per unit (a ring) and on one (a launch per slots)."""
import ctypes
import importlib

import pytest
import torch

from helpers import TOL, assert_close, to_dev
from test_mlp_bwd_gpu import GRADS, run_case
from test_mlp_fwd_gpu import mlp_case

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def P():
    return importlib.import_module("ttt-rs_amd")


@pytest.mark.parametrize("B,H,d,K,N,sg", [(1, 2, 32, 16, 2, True), (1, 1, 64, 16, 4, False), (1, 2, 96, 11, 19, True),
                                          (1, 1, 96, 16, 64, False), (2, 5, 64, 16, 33, True)])
def test_register_resident_backward(P, B, H, d, K, N, sg):
    print(f"case mlp bwd rp B{B} H{H} d{d} K{K} N{N} sg={sg}", flush=True)
    got, ref = run_case(P, B, H, d, K, N, torch.bfloat16, "baseline", sg)
    one, _ = run_case(P, B, H, d, K, N, torch.bfloat16, "baseline", sg, kernel_hint=P.TTT_HINT_ONE_WORKGROUP)
    for k in GRADS:
        # The usual bars: long sequences of one or two units leave up to 4 % of d_b1 outside the elementwise band, as they do
        # with the scan on tiles in memory.  d_token_eta is a sum over units with alternating signs: after two mini-batches
        # little but rounding is left of it (that scan misses it by 0.10 and has 31 % outside).
        few = k == "d_token_eta" and N == 2
        assert_close(got[k], ref[k], TOL[torch.bfloat16] * (5 if few else 1.25 if k == "d_token_eta" else 1), k,
                     min_frac=0.65 if few else 0.95)
        if k in ("d_token_eta", "d_gamma", "d_beta"):  # atomic additions: their order is not fixed
            assert_close(one[k], got[k].double(), 1e-5, k)
        else:
            assert torch.equal(one[k], got[k]), f"{k}: one workgroup per unit differs from two"


def saving_pair(P, v, d_out, K, fwd_hint, bwd_hint):
    a = (v["xq"], v["xk"], v["xv"], v["W1"], v["b1"], v["W2"], v["b2"], v["token_eta"], v["lr"], v["gamma"], v["beta"])
    saved = P.ttt_mlp_forward_raw(*a, K, kernel_hint=fwd_hint, save_for_backward=True)[5]
    return (P.ttt_mlp_backward_raw(*a, d_out, K, kernel_hint=bwd_hint, saved=saved),
            P.ttt_mlp_backward_raw(*a, d_out, K, kernel_hint=bwd_hint))


@pytest.mark.parametrize("d", [32, 96])
@pytest.mark.parametrize("fwd,bwd", [(f, b) for f in ("", "F32_PRODUCTS", "LDS_TILES") for b in ("", "F32_PRODUCTS", "LDS_TILES")])
def test_saved_buffer_says_which_form_it_has(P, fwd, bwd, d):
    """Whatever hint the saving forward had, the backward's results are those of the call that saves nothing: the forms
    of the saved factors differ between the kernels that the hints choose."""
    print(f"case mlp saving pair, forward hint {fwd or 'none'}, backward hint {bwd or 'none'}, d{d}", flush=True)
    K, N = 16, 5
    c = mlp_case(P, 555 + d, 1, 2, N * K, d, K, torch.bfloat16, "baseline")
    d_out = torch.randn(1, 2, N * K, d, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).to("cuda:0")
    hint = lambda name: getattr(P, "TTT_HINT_" + name) if name else 0
    got, ref = saving_pair(P, to_dev(c), d_out, K, hint(fwd), hint(bwd))
    torch.cuda.synchronize()
    for k in GRADS:
        if k in ("d_token_eta", "d_gamma", "d_beta"):  # atomic additions: their order is not fixed
            assert_close(got[k], ref[k].double(), 1e-5, k)
        else:
            assert torch.equal(got[k], ref[k]), k


def off_by_one(t):
    """The same contiguous tensor, one element behind a 16-byte boundary."""
    return torch.empty(t.numel() + 1, dtype=t.dtype, device="cuda:0")[1:].view(t.shape).copy_(t)


@pytest.mark.parametrize("save", [False, True])
@pytest.mark.parametrize("which", ["xq", "d_out", "d_xk", "d_W2", "all"])
def test_backward_takes_tensors_off_a_16_byte_boundary(P, which, save):
    """The kernels that move rows 16 bytes at a time give way to those that read element by element: to the scan with f32
    products, and where the rows of the forward are off to the sweep on LDS tiles as well."""
    print(f"case mlp bwd, unaligned {which}, saved {save}", flush=True)
    B, H, d, K, N = 1, 2, 64, 16, 4
    c = mlp_case(P, 611, B, H, N * K, d, K, torch.bfloat16, "baseline")
    d_out = torch.randn(B, H, N * K, d, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16)
    v = to_dev(c)
    names = ("xq", "xk", "xv", "W1", "b1", "W2", "b2", "token_eta", "lr", "gamma", "beta")
    a = [v[k] for k in names]
    hint = P.TTT_HINT_LDS_TILES if which in ("xq", "all") else P.TTT_HINT_F32_PRODUCTS
    ref = P.ttt_mlp_backward_raw(*a, d_out.to("cuda:0"), K, kernel_hint=hint)
    saved = P.ttt_mlp_forward_raw(*a, K, save_for_backward=True)[5] if save else None
    off = lambda k, t: off_by_one(t) if which in (k, "all") else t
    into = {k: off(k, torch.full_like(t, float("nan"))) for k, t in ref.items()}
    a = [off(k, t) if k in ("xq", "xk", "xv") else t for k, t in zip(names, a)]
    got = P.ttt_mlp_backward_raw(*a, off("d_out", d_out.to("cuda:0")), K, into=into, saved=saved)
    torch.cuda.synchronize()
    for k in GRADS:
        if k in ("d_token_eta", "d_gamma", "d_beta"):  # atomic additions: their order is not fixed
            assert_close(got[k], ref[k].double(), 1e-5, k)
        else:
            assert torch.equal(got[k], ref[k]), k


def test_static_scratch_takes_what_the_other_scan_fits(P):
    """On one workgroup per unit the register-resident scan needs more scratch than the scan with f32 products for
    sequences of a few mini-batches: a call whose scratch holds only the latter runs that."""
    B, H, d, K, N = 1, 57, 96, 16, 1
    print(f"case mlp bwd static B{B} H{H} d{d} N{N}", flush=True)
    hint = P.TTT_HINT_ONE_WORKGROUP
    desc = P.TttDesc(B, H, N * K, d, K, 1e-6, 1, P.TTT_BF16, 0, 0, 0, hint)
    assert P.lib().ttt_mlp_bwd_workspace_bytes(ctypes.byref(desc)) > 32 << 20
    v = to_dev(mlp_case(P, 613, B, H, N * K, d, K, torch.bfloat16, "baseline"))
    a = [v[k] for k in ("xq", "xk", "xv", "W1", "b1", "W2", "b2", "token_eta", "lr", "gamma", "beta")]
    d_out = torch.randn(B, H, N * K, d, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).to("cuda:0")
    got = P.ttt_mlp_backward_raw(*a, d_out, K, kernel_hint=hint, static_scratch=True)
    ref = P.ttt_mlp_backward_raw(*a, d_out, K, kernel_hint=hint | P.TTT_HINT_F32_PRODUCTS)
    torch.cuda.synchronize()
    for k in GRADS:
        if k in ("d_token_eta", "d_gamma", "d_beta"):  # atomic additions: their order is not fixed
            assert_close(got[k], ref[k].double(), 1e-5, k)
        else:
            assert torch.equal(got[k], ref[k]), k


@pytest.mark.parametrize("B,H,d,N", [(8, 16, 32, 96), (1, 8, 96, 40)])
def test_hand_over_slots_are_read_fresh(P, B, H, d, N):
    """Many turns of the ring of slots, up to as many units as run on two workgroups: what the consumer reads is what the
    producer stored this time, not what an earlier turn left in the consumer's vector cache (one workgroup per unit runs
    the two sides as separate launches)."""
    K = 16
    print(f"case mlp bwd rp ring B{B} H{H} d{d} N{N}", flush=True)
    v = to_dev(mlp_case(P, 612, B, H, N * K, d, K, torch.bfloat16, "baseline"))
    a = [v[k] for k in ("xq", "xk", "xv", "W1", "b1", "W2", "b2", "token_eta", "lr", "gamma", "beta")]
    d_out = torch.randn(B, H, N * K, d, generator=torch.Generator().manual_seed(8)).to(torch.bfloat16).to("cuda:0")
    got = P.ttt_mlp_backward_raw(*a, d_out, K)
    one = P.ttt_mlp_backward_raw(*a, d_out, K, kernel_hint=P.TTT_HINT_ONE_WORKGROUP)
    torch.cuda.synchronize()
    for k in GRADS:
        if k in ("d_token_eta", "d_gamma", "d_beta"):  # atomic additions: their order is not fixed
            assert_close(got[k], one[k].double(), 1e-4, k)
        else:
            assert torch.equal(got[k], one[k]), k
