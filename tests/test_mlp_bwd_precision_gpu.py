"""What the register-resident TTT-MLP backward (bf16 I/O) holds and multiplies in f32, element by element.

One mini-batch, no gradient of the output and one element of an upstream state gradient: the last token's d_token_eta is
then -lr * G1 * S1 (or G2 * S2) of a single token and hidden unit (or feature), the product of two numbers, and every matrix
operand behind it is exact in bf16 or rounded in the expectation too."""
import importlib
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

K, H_UNIT, F0, F1, TOK = 16, 5, 3, 17, 15  # tokens; the hidden unit, the features and the token that carry everything


@pytest.fixture(scope="module")
def P():
    return importlib.import_module("ttt-rs_amd")


def bf16(x):
    return x.to(torch.bfloat16).to(x.dtype)


def gelu_d(x):
    """tanh-GELU and its derivative in float64"""
    x = torch.as_tensor(x, dtype=torch.float64)
    c = math.sqrt(2 / math.pi)
    u = c * (x + 0.044715 * x**3)
    return x * torch.sigmoid(2 * u), torch.sigmoid(2 * u) + 0.5 * x / torch.cosh(u) ** 2 * c * (1 + 3 * 0.044715 * x * x)


def d_token_eta(P, d, x, through, seed=0):
    """The last token's d_token_eta with b1 = x, and what it is in float64 (G1, S1 or G2, S2 and their product)."""
    m = 4 * d
    g = torch.Generator().manual_seed(seed + d)
    xk, xv = torch.randn(1, 1, K, d, generator=g), torch.randn(1, 1, K, d, generator=g)
    xk, xv = xk.bfloat16(), xv.bfloat16()
    lr = torch.zeros(1, 1, K, dtype=torch.bfloat16)
    lr[0, 0, TOK] = 2.0**-7
    b2 = torch.randn(1, d, generator=g)
    W2 = torch.zeros(1, m, d)
    W2[0, H_UNIT, F0], W2[0, H_UNIT, F1] = 0.375, -0.375  # row mean 0: the kernels carry W2 centred
    b1 = torch.full((1, m), float(x))
    up = [torch.zeros(1, 1, d, m), torch.zeros(1, 1, m), torch.zeros(1, 1, m, d), torch.zeros(1, 1, d)]
    if through == "G1":
        up[0][0, 0, :, H_UNIT] = 0.25
    else:
        up[2][0, 0, H_UNIT, F0] = 0.75
    dev = lambda t: t.to("cuda:0")
    te = 1.0 / torch.arange(1, K + 1, dtype=torch.float32)
    got = P.ttt_mlp_backward_raw(dev(xk), dev(xk), dev(xv), dev(torch.zeros(1, d, m)), dev(b1), dev(W2), dev(b2), dev(te),
                                 dev(lr), dev(torch.ones(1, d)), dev(torch.zeros(1, d)),
                                 dev(torch.zeros(1, 1, K, d, dtype=torch.bfloat16)), K, d_state_out=[dev(t) for t in up])
    torch.cuda.synchronize()
    y, dy = gelu_d(b1[0, H_UNIT].item())
    x2 = bf16(y)
    z = x2 * W2[0, H_UNIT].double() + b2[0].double()
    rstd = (z.var(unbiased=False) + 1e-6) ** -0.5
    xh = (z - z.mean()) * rstd
    t = xv[0, 0, TOK].double() - xk[0, 0, TOK].double()
    gx = xh - t
    G2 = (gx - gx.mean() - xh * (gx * xh).mean()) * rstd
    U = (bf16(G2) * W2[0, H_UNIT].double()).sum()
    if through == "G1":
        a, s = U * dy, xk[0, 0, TOK].double().sum() * 0.25
    else:
        a, s = G2[F0], x2 * 0.75
    return got["d_token_eta"][K - 1].item(), -(2.0**-7) * (a * s).item(), (U * s).item() * 2.0**-7


@pytest.mark.parametrize("d", [32, 64, 96])
def test_g2_enters_d_lr_unrounded(P, d):
    """X2 : T2, the kernel's form of G2 : S2, takes G2 in two bf16 parts: it may miss 2^-17 of it (two parts of 8 bits and
    a sign), and the f32 products beside it."""
    for seed in range(6):
        print(f"case G2 in d_token_eta, d{d} seed {seed}", flush=True)
        got, ref, _ = d_token_eta(P, d, 1.0, "G2", seed)
        assert abs(got - ref) <= 2.0**-16 * abs(ref), (got, ref)


@pytest.mark.parametrize("d", [32, 64, 96])
def test_g1_enters_d_lr_in_f32(P, d):
    """An operand's rounding would be up to 2^-9 of G1; f32 products and a sum of d terms of one size leave 2^-14 even where
    the sum nearly cancels."""
    for seed in range(6):
        print(f"case G1 in d_token_eta, d{d} seed {seed}", flush=True)
        got, ref, _ = d_token_eta(P, d, 0.0, "G1", seed)
        assert abs(got - ref) <= 2.0**-14 * abs(ref), (got, ref)


def test_gelu_derivative_is_as_good_as_the_tanh_form(P):
    """gelu'(x) = G1 / U where its terms cancel (x from -4.5 to -1.5), against float64: the error may be that of the tanh
    form in float32 with a correctly rounded tanh, computed here at the same points, and half of it more for the products
    around it.  (1 + tanh through exp2 and rcp, without a tanh, has 2.6 times that error.)"""
    print("case gelu' through d_token_eta", flush=True)
    c = math.sqrt(2 / math.pi)
    err, ref = 0.0, 0.0
    for i in range(40):
        x = torch.tensor(-4.5 + 3.0 * (i + 0.37) / 40, dtype=torch.float32)
        got, _, scale = d_token_eta(P, 32, x.item(), "G1", 1)
        dy = gelu_d(x.item())[1].item()
        t = torch.tanh((c * (x + 0.044715 * x * x * x)).double()).float()
        f32 = 0.5 * (1 + t) + 0.5 * x * (1 - t * t) * c * (1 + 3 * 0.044715 * x * x)
        err += (-got / scale - dy) ** 2
        ref += (f32.double().item() - dy) ** 2
    print(f"rms error {math.sqrt(err / 40):.3e}, of the tanh form in float32 {math.sqrt(ref / 40):.3e}")
    assert err <= 1.5**2 * ref


def one_mini_batch(c, rnd):
    """d_xv and d_lr of a mini-batch from float64 products of operands that went through rnd (identity or a bf16 rounding),
    each operand rounded once and the same one in every product that takes it; per unit, [U, ...]."""
    T = lambda t: t.transpose(-1, -2)
    xq, xk, xv, dO, te, lr = (c[k].double() for k in ("xq", "xk", "xv", "d_out", "token_eta", "lr"))
    W1, W2 = rnd(c["W1"].double()), rnd(c["W2"].double())
    causal = torch.tril(torch.ones(K, K, dtype=torch.float64))

    def norm(z):
        r = (z.var(-1, unbiased=False, keepdim=True) + 1e-6) ** -0.5
        return (z - z.mean(-1, keepdim=True)) * r, r

    def norm_bwd(g, xh, r):
        return (g - g.mean(-1, keepdim=True) - xh * (g * xh).mean(-1, keepdim=True)) * r

    x2, g1 = gelu_d(xk @ W1)
    x2 = rnd(x2)
    xh, rstd = norm(x2 @ W2)
    G2 = rnd(norm_bwd(xh - (xv - xk), xh, rstd))
    G1 = rnd(G2 @ T(W2) * g1)
    eta = te[:, None] * lr[:, None, :] * causal
    A1 = xq @ T(xk)
    M1 = rnd(eta * (1 + A1))
    xb2, gb1 = gelu_d(xq @ W1 - M1 @ G1)
    xb2 = rnd(xb2)
    A2 = xb2 @ T(x2)
    M2 = rnd(eta * (1 + A2))
    xhb, rb = norm(xb2 @ W2 - M2 @ G2)
    dz2 = rnd(norm_bwd(dO, xhb, rb))
    P2 = dz2 @ T(G2) * causal
    dz1 = rnd((dz2 @ T(W2) + rnd(-P2 * eta) @ x2) * gb1)
    P1 = dz1 @ T(G1) * causal
    d_lr = (-(P2 * (1 + A2) + P1 * (1 + A1)) * te[:, None]).sum(-2)
    u = (T(M2) @ dz2 - rnd(-(T(M1) @ dz1) * g1) @ W2) * rstd
    return u - u.mean(-1, keepdim=True) - xh * (u * xh).mean(-1, keepdim=True), d_lr


def test_an_operand_is_rounded_once_for_all_products(P):
    """G1, G2 and the causal blocks enter the forward's intermediates and the gradient's products.  Rounded anew in each
    (as products with the learning rate, say) they make d_xv worse by 8 % and d_lr by 10 - 18 %: the errors against float64
    are held to those of float64 products of operands rounded once, within what 64 units of one mini-batch scatter."""
    print("case operand roundings, 64 units of d64", flush=True)
    B, H, d = 4, 16, 64
    U, m = B * H, 4 * d
    g = torch.Generator().manual_seed(21)
    n = lambda *s: torch.randn(*s, generator=g)
    c = {k: n(U, K, d).bfloat16() for k in ("xq", "xk", "xv", "d_out")}
    c.update(W1=0.02 * n(U, d, m), W2=0.02 * n(U, m, d), lr=(torch.sigmoid(n(U, K)) / d).bfloat16(),
             token_eta=1.0 / torch.arange(1, K + 1, dtype=torch.float32))
    dev = lambda t, *s: t.reshape(B, H, *s).to("cuda:0")
    z = lambda *s: torch.zeros(*s, device="cuda:0")
    got = P.ttt_mlp_backward_raw(*(dev(c[k], K, d) for k in ("xq", "xk", "xv")), dev(c["W1"], d, m), z(B, H, m),
                                 dev(c["W2"], m, d), z(B, H, d), c["token_eta"].to("cuda:0"), dev(c["lr"], K), z(H, d) + 1,
                                 z(H, d), dev(c["d_out"], K, d), K)
    torch.cuda.synchronize()
    exact, once = one_mini_batch(c, lambda t: t), one_mini_batch(c, bf16)
    for name, e, o in zip(("d_xv", "d_lr"), exact, once):
        e, o, r = e.flatten(), bf16(o).flatten(), got[name].cpu().double().flatten()
        err, expected = (r - e).norm().item(), (o - e).norm().item()
        print(f"{name}: relative error {err / e.norm().item():.3e}, with operands rounded once {expected / e.norm().item():.3e}")
        assert err <= 1.04 * expected, name
