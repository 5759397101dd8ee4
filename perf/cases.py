"""The inner-loop work that a user of this package has it do, as cases that can be timed and compared.

A case names a kind of call and its sizes; the sizes are those of bench.py's workloads (H = 12, d = 64: the 125M shape;
H = 16 with d = 96 or 128: the TTT-MLP and the long-context shapes) and generic ones around them.  `prepare` makes what a
program holds before the call, `run` is one pass through the package's public entry points.
"""
import ctypes
import importlib

import torch

pkg = importlib.import_module("ttt-rs_amd")

DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}
K = 16  # tokens of a mini-batch


def listed():
    return [
        # Generation: the next few tokens of one sequence on a state that is carried from call to call, each layer of a
        # model once per step.  Latency: one short launch and the host path in front of it.
        {"name": "linear_decode_bf16", "kind": "decode", "io": "bf16", "B": 1, "H": 12, "d": 64, "seq": 16},
        # A prompt of any length into the layer object: whole mini-batches and a short one at the end, f32 activations.
        {"name": "linear_prompt_f32", "kind": "prompt", "io": "f32", "B": 2, "H": 12, "d": 64, "seq": 1013},
        # Inference on a large batch at the 125M shape: the benchmark's headline forward.
        {"name": "linear_fwd_bf16", "kind": "linear_fwd", "io": "bf16", "B": 32, "H": 12, "d": 64, "seq": 2048},
        # A training step at the 125M shape with bf16 activations, in the checkpoint format the library recommends.
        {"name": "linear_train_bf16", "kind": "linear_train", "io": "bf16", "B": 32, "H": 12, "d": 64, "seq": 2048, "ci": 1},
        # The same with f32 activations and a smaller batch.
        {"name": "linear_train_f32", "kind": "linear_train", "io": "f32", "B": 8, "H": 12, "d": 64, "seq": 2048, "ci": 1},
        # Training with a state saved every 16 mini-batches only: what a caller short of memory asks for.
        {"name": "linear_train_sparse_f32", "kind": "linear_train", "io": "f32", "B": 8, "H": 12, "d": 64, "seq": 2048,
         "ci": 16},
        # A layer from its projections to its output projection: head split, rotary embedding, lr gate, inner loop,
        # head merge, norm and gate.
        {"name": "linear_layer_bf16", "kind": "layer", "io": "bf16", "B": 32, "H": 12, "d": 64, "seq": 2048},
        # Inference with the TTT-MLP inner model.
        {"name": "mlp_fwd_bf16", "kind": "mlp_fwd", "io": "bf16", "B": 8, "H": 16, "d": 96, "seq": 2048},
        # A training step with it: the forward that saves and the backward that uses what was saved.
        {"name": "mlp_train_bf16", "kind": "mlp_train", "io": "bf16", "B": 8, "H": 16, "d": 96, "seq": 2048},
        # Long context: six TTT-Linear and two TTT-MLP layers as one call, in windows of 2048 tokens on two streams.
        {"name": "stack_bf16", "kind": "stack", "io": "bf16", "B": 4, "H": 16, "d": 128, "seq": 8192, "linear": 6, "mlp": 2,
         "chunk": 2048},
        # The other inner models, a batch of sequences forward: TTT-Linear with the Adam inner optimiser ...
        {"name": "adam_fwd_bf16", "kind": "adam", "io": "bf16", "B": 32, "H": 12, "d": 64, "seq": 2048},
        # ... and TTT-MLP with two hidden layers.
        {"name": "mlp2_fwd_bf16", "kind": "mlpn", "io": "bf16", "B": 8, "H": 12, "d": 64, "seq": 1024, "hidden": 2},
    ]


def _spread(rng, lo, hi):
    """A whole number from lo to hi, even over its logarithm."""
    return min(hi, int(lo * ((hi + 1) / lo) ** rng.random()))


def _tokens(rng, lo, hi):
    """A sequence length of whole mini-batches."""
    return K * _spread(rng, -(-lo // K), hi // K)


def draw(rng):
    kind = rng.choice(["decode", "prompt", "linear_fwd", "linear_train", "linear_train", "linear_train_sparse", "layer",
                       "mlp_fwd", "mlp_train", "stack", "adam", "mlpn"])
    io = rng.choice(["bf16", "f32"])
    H = rng.choice([4, 8, 12, 16])
    if kind == "decode":  # one step of up to a mini-batch for one or for many sequences
        return {"kind": kind, "io": io, "B": _spread(rng, 1, 64), "H": H, "d": rng.choice([32, 64, 64, 96, 128]),
                "seq": rng.randint(1, K)}
    if kind == "prompt":
        return {"kind": kind, "io": io, "B": _spread(rng, 1, 8), "H": H, "d": rng.choice([32, 64, 64, 128]),
                "seq": _spread(rng, 17, 2048)}
    if kind == "linear_fwd":
        return {"kind": kind, "io": io, "B": _spread(rng, 1, 32), "H": H, "d": rng.choice([32, 64, 64, 96, 128]),
                "seq": _tokens(rng, 64, 2048)}
    if kind == "linear_train":
        return {"kind": kind, "io": io, "B": _spread(rng, 1, 32 if io == "bf16" else 16), "H": H,
                "d": rng.choice([32, 64, 64]), "seq": _tokens(rng, 64, 2048), "ci": 1}
    if kind == "linear_train_sparse":
        return {"kind": "linear_train", "io": io, "B": _spread(rng, 1, 8), "H": H, "d": rng.choice([32, 64, 64]),
                "seq": _tokens(rng, 64, 2048), "ci": rng.choice([2, 4, 8, 16])}
    if kind == "layer":
        return {"kind": kind, "io": "bf16", "B": _spread(rng, 1, 32), "H": H, "d": rng.choice([32, 64, 64]),
                "seq": _tokens(rng, 64, 2048)}
    if kind == "mlp_fwd":
        return {"kind": kind, "io": "bf16", "B": _spread(rng, 1, 8), "H": H, "d": rng.choice([64, 96, 96, 128]),
                "seq": _tokens(rng, 64, 2048)}
    if kind == "mlp_train":
        return {"kind": kind, "io": "bf16", "B": _spread(rng, 1, 8), "H": H, "d": rng.choice([64, 96, 96]),
                "seq": _tokens(rng, 64, 2048)}
    if kind == "stack":
        chunk = rng.choice([512, 1024, 2048])
        return {"kind": kind, "io": "bf16", "B": _spread(rng, 1, 4), "H": rng.choice([8, 12, 16]), "d": rng.choice([64, 128]),
                "seq": chunk * rng.randint(1, 8192 // chunk), "linear": rng.randint(1, 6), "mlp": rng.randint(0, 2),
                "chunk": chunk}
    if kind == "adam":
        return {"kind": kind, "io": io, "B": _spread(rng, 1, 32), "H": H, "d": rng.choice([32, 64, 64]),
                "seq": _tokens(rng, 64, 2048)}
    hidden, d = rng.choice([(2, 32), (3, 32), (4, 32), (2, 64), (2, 64), (2, 64)])
    return {"kind": kind, "io": io, "B": _spread(rng, 1, 8), "H": H, "d": d, "seq": _tokens(rng, 64, 1024), "hidden": hidden}


class _Draws:
    """Seeded tensors on the device, with the distributions of the benchmark's inputs."""

    def __init__(self, case, seed):
        self.dev = torch.device("cuda")
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(int(seed))
        self.B, self.H, self.d, self.seq = case["B"], case["H"], case["d"], case["seq"]
        self.io = DTYPES[case["io"]]

    def normal(self, *shape, scale=1.0, dtype=torch.float32):
        t = torch.randn(*shape, generator=self.g, dtype=dtype, device=self.dev)
        return t if scale == 1.0 else t.mul_(scale)

    def rows(self):
        return self.normal(self.B, self.H, self.seq, self.d, dtype=self.io)

    def gates(self):
        """ttt_lr_eta: base_lr / d times the sigmoid of N(0, 1) logits."""
        return (torch.sigmoid(self.normal(self.B, self.H, self.seq)) / self.d).to(self.io)

    def norm(self):
        return torch.ones(self.H, self.d, device=self.dev), torch.zeros(self.H, self.d, device=self.dev)

    def weights(self, n_in, n_out):
        return self.normal(self.H, n_in, n_out, scale=0.02), torch.zeros(self.H, n_out, device=self.dev)

    def token_eta(self, n):
        return (1.0 / torch.arange(1, K + 1, dtype=torch.float32, device=self.dev)).repeat(-(-n // K))[:n].contiguous()


def prepare(case, seed):
    r = _Draws(case, seed)
    kind, B, H, d, seq = case["kind"], r.B, r.H, r.d, r.seq
    s = {"kind": kind, "B": B}
    s["ln"] = r.norm()
    if kind in ("decode", "prompt"):
        W, b = r.weights(d, d)
        s["layer"] = pkg.FusedTileMulti(pkg.ModelConfig(H, d, pkg.TTTConfig(mini_batch_size=K)), W, b, *s["ln"])
        s["inputs"] = pkg.TTTInputsInner(pkg.Qkv(r.rows(), r.rows(), r.rows()), r.token_eta(seq), r.gates())
        if kind == "decode":  # a state that has seen a prompt
            s["state"] = (r.normal(B, H, d, d, scale=0.02), r.normal(B, H, d, scale=0.02))
            s["range"] = range(0, seq)
    elif kind == "layer":
        s["x"] = [r.normal(B, seq, H, d, dtype=r.io) for _ in range(3)]
        s["logits"] = r.normal(B, seq, H, dtype=r.io)
        s["lr_bias"] = torch.zeros(H, device=r.dev)
        s["token_idx"], s["learnable"] = r.token_eta(K), torch.zeros(K, device=r.dev)
        s["rope"] = pkg.rope_cos_sin(K, 0, None, d, r.dev)
        s["W"], s["b"] = r.weights(d, d)
        s["post"] = torch.ones(H * d, device=r.dev), torch.zeros(H * d, device=r.dev)
        s["gate"] = r.normal(B, seq, H * d, dtype=r.io)
    elif kind == "stack":
        s["te"], s["chunk"], s["layers"] = r.token_eta(K), case["chunk"], []
        for i in range(case["linear"] + case["mlp"]):
            L = {"pq": r.rows(), "pk": r.rows(), "pv": r.rows(), "lr": r.gates()}
            L["gamma"], L["beta"] = r.norm()
            if i < case["linear"]:
                L["W0"], L["b0"] = r.weights(d, d)
            else:
                L["W1"], L["b1"] = r.weights(d, 4 * d)
                L["W2"], L["b2"] = r.weights(4 * d, d)
            s["layers"].append(L)
        n = pkg.ttt_stack_workspace_bytes(B, H, seq, d, K, r.io, [i >= case["linear"] for i in range(len(s["layers"]))],
                                          s["chunk"])
        s["workspace"] = torch.empty(n, dtype=torch.uint8, device=r.dev)
        s["aux"] = torch.cuda.Stream(r.dev)
    else:
        s["x"] = [r.rows(), r.rows(), r.rows()]
        s["eta"] = (r.token_eta(K), r.gates())
        if kind in ("linear_fwd", "linear_train", "adam"):
            s["W"], s["b"] = r.weights(d, d)
        elif kind in ("mlp_fwd", "mlp_train"):
            s["W"], s["b"], s["W2"], s["b2"] = r.weights(d, 4 * d) + r.weights(4 * d, d)
        else:
            dims = [d] + [4 * d] * case["hidden"] + [d]
            wb = [r.weights(dims[i], dims[i + 1]) for i in range(case["hidden"] + 1)]
            s["W"], s["b"] = [w for w, _ in wb], [b for _, b in wb]
        if kind in ("linear_train", "mlp_train"):
            s["d_out"] = r.rows()
        if kind == "linear_train":
            s["ci"] = case["ci"]
            desc = pkg.TttDesc(B, H, seq, d, K, 1e-6, case["ci"], pkg.TTT_BF16 if case["io"] == "bf16" else pkg.TTT_F32)
            s["format"] = pkg.lib().ttt_linear_best_checkpoint_format(ctypes.byref(desc))
    return s


def run(s):
    kind = s["kind"]
    if kind == "decode":
        state = pkg.TTTLinearState(*s["state"])
        out = s["layer"].forward_mini_batch(state, s["inputs"], s["range"])
        return out, state.weight, state.bias
    if kind == "prompt":
        state = s["layer"].init_state(s["B"])
        out = s["layer"].forward(state, s["inputs"])
        return out, state.weight, state.bias
    if kind == "layer":
        out, W, b = pkg.ttt_linear_forward_fused_inputs_raw(*s["x"], s["logits"], s["lr_bias"], 1.0, s["token_idx"],
                                                            s["learnable"], s["W"], s["b"], *s["ln"], K, rope=s["rope"],
                                                            pos_wrap=K)
        return pkg.layer_epilogue_raw(out, *s["post"], gate=s["gate"]), W, b
    if kind == "stack":
        return pkg.ttt_stack_forward_raw(s["layers"], s["te"], K, workspace=s["workspace"], chunk_tokens=s["chunk"],
                                         aux_stream=s["aux"], check_lost=False)
    if kind == "linear_fwd":
        return pkg.ttt_linear_forward_raw(*s["x"], s["W"], s["b"], *s["eta"], *s["ln"], K)
    if kind == "linear_train":
        a = (*s["x"], s["W"], s["b"], *s["eta"], *s["ln"])
        out, W, b, W_ckpt, b_ckpt = pkg.ttt_linear_forward_raw(*a, K, checkpoint_interval=s["ci"], want_checkpoints=True,
                                                               packed_checkpoints=s["format"])
        g = pkg.ttt_linear_backward_raw(*a, W_ckpt, b_ckpt, s["d_out"], K, checkpoint_interval=s["ci"],
                                        packed_checkpoints=s["format"])
        return out, W, b, g
    if kind == "adam":
        return pkg.ttt_linear_adam_forward_raw(*s["x"], s["W"], s["b"], *s["eta"], *s["ln"], K)
    if kind == "mlpn":
        return pkg.ttt_mlpn_forward_raw(*s["x"], s["W"], s["b"], *s["eta"], *s["ln"], K)
    a = (*s["x"], s["W"], s["b"], s["W2"], s["b2"], *s["eta"], *s["ln"])
    if kind == "mlp_fwd":
        return pkg.ttt_mlp_forward_raw(*a, K)
    out, W1, b1, W2, b2, saved = pkg.ttt_mlp_forward_raw(*a, K, save_for_backward=True)
    return out, W1, b1, W2, b2, pkg.ttt_mlp_backward_raw(*a, s["d_out"], K, saved=saved)


def work(case):
    """Per token of one head: the operands read and the results written once, and the products of the dual form with
    causal blocks of a mini-batch; the states besides, read once per head and written once per sequence and head."""
    B, H, d, seq, kind = case["B"], case["H"], case["d"], case["seq"], case["kind"]
    n, s = B * H * seq, 2 if case["io"] == "bf16" else 4
    linear, mlp = d * d + d, 8 * d * d + 5 * d
    lin_flops, mlp_flops = 6 * d * d + 4 * K * d, 56 * d * d + 20 * K * d
    fwd = n * (4 * d * s + s)
    if kind in ("decode", "prompt"):
        return {"bytes": fwd + 4 * linear * H * ((B if kind == "decode" else 1) + B), "flops": n * lin_flops}
    if kind == "linear_fwd":
        return {"bytes": fwd + 4 * linear * H * (1 + B), "flops": n * lin_flops}
    if kind == "layer":  # three projections and the gate in, one tensor out
        return {"bytes": n * (5 * d * s + s) + 4 * linear * H * (1 + B), "flops": n * lin_flops}
    if kind == "linear_train":
        return {"bytes": n * (11 * d * s + 3 * s) + 4 * linear * H * (2 + 2 * B), "flops": n * (24 * d * d + 26 * K * d)}
    if kind == "mlp_fwd":
        return {"bytes": fwd + 4 * mlp * H * (1 + B), "flops": n * mlp_flops}
    if kind == "mlp_train":
        return {"bytes": n * (11 * d * s + 3 * s) + 4 * mlp * H * (2 + 2 * B), "flops": n * (224 * d * d + 80 * K * d)}
    if kind == "stack":  # three projections of every layer in; the hand-over between layers need not leave the chip
        layers = case["linear"] + case["mlp"]
        return {"bytes": n * (layers * (3 * d * s + s) + d * s) + 4 * H * (1 + B) * (case["linear"] * linear + case["mlp"] * mlp),
                "flops": n * (case["linear"] * lin_flops + case["mlp"] * mlp_flops)}
    if kind == "adam":  # three f32 tensors of state; about ten operations an element and mini-batch for the step
        return {"bytes": fwd + 4 * linear * H * (1 + 3 * B), "flops": n * lin_flops + n // K * 10 * linear}
    dims = [d] + [4 * d] * case["hidden"] + [d]
    params = sum(a * b for a, b in zip(dims, dims[1:]))
    return {"bytes": fwd + 4 * (params + sum(dims[1:])) * H * (1 + B),
            "flops": n * (8 * params - 8 * d * d + 4 * K * sum(a + b for a, b in zip(dims, dims[1:])))}


def tolerance(case):
    """What the package promises its callers, 1e-4 for f32 activations; for bf16 ones an operand's rounding (2^-9) goes
    through a recurrence over the whole sequence.  Gradients with bf16 activations are also sums of terms that largely
    cancel.  An Adam step has the size of its rate whatever the gradient's: an element whose gradient is all rounding may
    go the other way."""
    rel = 1e-4 if case["io"] == "f32" else 2e-2 if case["kind"] in ("linear_train", "mlp_train") else 1e-2
    if case["kind"] == "adam":
        return {"rel": rel, "max": 0.5}
    return {"rel": rel}
