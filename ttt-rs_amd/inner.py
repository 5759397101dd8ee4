"""Host-side mirror of the reference's inner-model interface for the fused TTT-Linear layer.

Names and argument meaning follow the reference:
  TTTInnerModel trait            rust/core/src/inner.rs:13-58
  Qkv / TTTInputsInner           rust/core/src/inner.rs:60-130
  TTTLinear / TTTLinearState     rust/core/src/linear.rs:17-89
  Fused<_, TTTLinear, TileMultiKernel> ("fused-tile-multi")
                                 rust/fused/src/linear_fused_tile/wrapper.rs:81-211
All arithmetic happens in the HIP library behind include/ttt_mi355x.h.
"""
from __future__ import annotations

import ctypes as C
from dataclasses import dataclass, field
from typing import Optional

import torch

from . import _lib
from ._lib import TttDesc, check, host, lib


@dataclass
class TTTConfig:
    """Subset of rust/config/src/train.rs:11-141 used by the inner loop."""
    mini_batch_size: int = 16
    base_lr: float = 1.0
    epsilon: float = 1e-6
    checkpoint_interval: int = 1
    mlp_expansion_factor: int = 4


@dataclass
class ModelConfig:
    num_heads: int
    head_dim: int
    ttt: TTTConfig = field(default_factory=TTTConfig)


@dataclass
class Qkv:
    """[batch, heads, seq, head_dim] each (inner.rs:60-68)."""
    xq: torch.Tensor
    xk: torch.Tensor
    xv: torch.Tensor

    def slice_seq(self, r: range) -> "Qkv":
        return Qkv(self.xq[:, :, r.start:r.stop], self.xk[:, :, r.start:r.stop], self.xv[:, :, r.start:r.stop])


@dataclass
class TTTInputsInner:
    """inner.rs:107-119. token_eta [seq] f32, ttt_lr_eta [batch, heads, seq]."""
    qkv: Qkv
    token_eta: torch.Tensor
    ttt_lr_eta: torch.Tensor
    start_idx: int = 0

    def slice_seq(self, r: range) -> "TTTInputsInner":
        return TTTInputsInner(self.qkv.slice_seq(r), self.token_eta[r.start:r.stop],
                              self.ttt_lr_eta[:, :, r.start:r.stop], r.start)


@dataclass
class TTTLinearState:
    """linear.rs:27-33: weight [B,H,d,d], bias [B,H,d], always f32."""
    weight: torch.Tensor
    bias: torch.Tensor


def _need(t: torch.Tensor, shape, dtype, name):
    if tuple(t.shape) != tuple(shape):
        raise _lib.TttError(_lib.TTT_ERR_SHAPE, f"{name}: shape {tuple(t.shape)} != {tuple(shape)}")
    if t.dtype != dtype:
        raise _lib.TttError(_lib.TTT_ERR_SHAPE, f"{name}: dtype {t.dtype} != {dtype}")
    if not t.is_cuda:
        raise _lib.TttError(_lib.TTT_ERR_NULL, f"{name} is not a device tensor")
    return t.contiguous()


def ttt_linear_forward_raw(xq, xk, xv, weight, bias, token_eta, ttt_lr_eta, ln_weight, ln_bias,
                           mini_batch: int, eps: float = 1e-6, checkpoint_interval: int = 1,
                           want_checkpoints: bool = False, out: Optional[torch.Tensor] = None, packed_checkpoints: bool = False,
                           kernel_hint: int = 0):
    """One call of ttt_linear_fwd on the current stream.

    Counterpart of fused_ttt_tile_forward_multi (rust/fused/src/linear_fused_tile/api.rs:52-83):
    weight [B,H,d,d] or [H,d,d], bias [B,H,d] or [H,d], token_eta [>=K] (first K entries used).
    Returns (output, weight_out, bias_out[, weight_ckpt, bias_ckpt]).
    packed_checkpoints is ttt_desc.checkpoint_format: False/0 f32 matrices; True/1 (interval 1) W checkpoints as
    operand fragments in kernel order; 2 (bf16 I/O, interval 1, d <= 96) the update factors and the final state
    instead of states.  The result is to be handed to ttt_linear_backward_raw with the same value; the tensors keep
    their f32 [B,H,n,d,d] / [B,H,n,d] allocations whatever the format.
    """
    return host().linear_forward(xq, xk, xv, weight, bias, token_eta, ttt_lr_eta, ln_weight, ln_bias, mini_batch, eps,
                                 checkpoint_interval, want_checkpoints, out, int(packed_checkpoints), kernel_hint)


def ttt_linear_adam_forward_raw(xq, xk, xv, weight, bias, token_eta, ttt_lr_eta, ln_weight, ln_bias, mini_batch: int,
                                beta1: float = 0.9, beta2: float = 0.999, adam_eps: float = 1e-8, adam_lr: float = 1e-3,
                                moments=None, step: int = 0, eps: float = 1e-6):
    """One call of ttt_linear_adam_fwd on the current stream: TTTLinearAdam::forward
    (rust/core/src/linear_adam.rs:183-236 looped as rust/core/src/inner.rs:25-50).  Arguments as
    ttt_linear_forward_raw; moments = (weight_m, bias_m, weight_v, bias_v) per batch element to continue an earlier call
    at `step`, or None for a fresh state.  Returns (output, weight, bias, (weight_m, bias_m, weight_v, bias_v), step)."""
    return host().linear_adam_forward(xq, xk, xv, weight, bias, token_eta, ttt_lr_eta, ln_weight, ln_bias, mini_batch,
                                      beta1, beta2, adam_eps, adam_lr, moments, int(step), eps)


def ttt_linear_backward_raw(xq, xk, xv, weight, bias, token_eta, ttt_lr_eta, ln_weight, ln_bias,
                            weight_ckpt, bias_ckpt, grad_output, mini_batch: int, eps: float = 1e-6,
                            checkpoint_interval: int = 1, grad_weight_out=None, grad_bias_out=None, packed_checkpoints: bool = False,
                            kernel_hint: int = 0, workspace=None):
    """One call of ttt_linear_bwd (or ttt_linear_bwd_ws, where the library has a kernel that uses a workspace: f32
    I/O up to 128 units runs every unit on two workgroups; with checkpoint_interval > 1 the states between the checkpoints
    are computed first, into up to 256 MiB) on the current stream.  workspace: a device tensor of
    ttt_linear_bwd_workspace_bytes(desc) bytes, None to allocate one for the call, False to call the entry point without
    (the memory of sparse checkpoints and nothing else, at several times the time).

    Counterpart of backward_multi (rust/fused/src/linear_fused_tile/backward/launch.rs:332-438).
    Returns a dict with the nine input gradients named as TttGradInputs
    (backward/launch.rs:427-437): grad_xq, grad_xk, grad_xv, grad_weight [B,H,d,d],
    grad_bias [B,H,d], grad_ttt_lr_eta, grad_token_eta [seq], grad_ln_weight, grad_ln_bias.
    """
    return host().linear_backward(xq, xk, xv, weight, bias, token_eta, ttt_lr_eta, ln_weight, ln_bias, weight_ckpt,
                                  bias_ckpt, grad_output, mini_batch, eps, checkpoint_interval, grad_weight_out,
                                  grad_bias_out, int(packed_checkpoints), kernel_hint, workspace)


def ttt_mlp_forward_raw(xq, xk, xv, w1, b1, w2, b2, token_eta, ttt_lr_eta, ln_weight, ln_bias,
                        mini_batch: int, eps: float = 1e-6, kernel_hint: int = 0, save_for_backward: bool = False):
    """One call of ttt_mlp_fwd on the current stream: the fused counterpart of
    TTTMLP::forward (rust/core/src/mlp.rs:127-208 looped as rust/core/src/inner.rs:25-50).
    w1 [B,H,d,4d] or [H,d,4d], b1 [..,4d], w2 [..,4d,d], b2 [..,d].
    Returns (output, w1_out, b1_out, w2_out, b2_out), state per batch element.
    save_for_backward: call ttt_mlp_fwd_saving instead and return a sixth element, the `saved` buffer that
    ttt_mlp_backward_raw(saved=...) consumes (the backward then skips its own forward sweep)."""
    return host().mlp_forward(xq, xk, xv, w1, b1, w2, b2, token_eta, ttt_lr_eta, ln_weight, ln_bias, mini_batch, eps,
                              kernel_hint, save_for_backward)


def ttt_mlpn_forward_raw(xq, xk, xv, weights, biases, token_eta, ttt_lr_eta, ln_weight, ln_bias, mini_batch: int,
                         eps: float = 1e-6, kernel_hint: int = 0):
    """One call of ttt_mlpn_fwd on the current stream: TTTMLP2/3/4::forward (rust/core/src/mlp2.rs, mlp3.rs, mlp4.rs
    looped as rust/core/src/inner.rs:25-50).  weights / biases: lists of the n_hidden + 1 layers, [H,in,out] / [H,out] or
    with a leading batch dimension.  Returns (output, weights_out, biases_out), state per batch element.
    kernel_hint: with at most half as many (batch, head) units as the device has CUs and four mini-batches or more a unit
    runs on two workgroups that wait for each other; TTT_HINT_ONE_WORKGROUP keeps it on one (the same bits), for a device
    that other work holds for seconds, where the wait would be in vain and the unit computed again on one workgroup."""
    return host().mlpn_forward(xq, xk, xv, list(weights), list(biases), token_eta, ttt_lr_eta, ln_weight, ln_bias,
                               mini_batch, eps, int(kernel_hint))


def ttt_mlp_backward_raw(xq, xk, xv, w1, b1, w2, b2, token_eta, ttt_lr_eta, ln_weight, ln_bias, d_out,
                         mini_batch: int, eps: float = 1e-6, d_state_out=None, static_scratch: bool = False,
                         into=None, kernel_hint: int = 0, saved=None):
    """One call of ttt_mlp_bwd on the current stream: gradients of the TTT-MLP inner loop
    (rust/core/src/mlp.rs:127-208 looped as rust/core/src/inner.rs:25-50; the reference gets them
    from Burn autodiff).  Arguments as ttt_mlp_forward_raw plus d_out [B,H,seq,d] and the optional
    upstream gradients of the final state d_state_out = (dW1, db1, dW2, db2), per batch element.
    Returns a dict: d_xq, d_xk, d_xv, d_W1 [B,H,d,4d], d_b1, d_W2, d_b2 (per batch element), d_lr,
    d_token_eta [seq], d_gamma, d_beta [H,d].
    static_scratch: call ttt_mlp_bwd_static (the library's built-in scratch buffer instead of a workspace
    allocated here); `into`: a dict returned by an earlier call of the same shape, whose tensors receive the
    gradients (with both, the call allocates no device memory).  kernel_hint: TTT_HINT_F32_PRODUCTS keeps the
    reverse scan's products in f32 where it would round their operands to bf16 (bf16 I/O, head_dim <= 96).
    saved: the buffer a forward with save_for_backward=True returned (same inputs, same hint): ttt_mlp_bwd_saved, which
    consumes it."""
    return host().mlp_backward(xq, xk, xv, w1, b1, w2, b2, token_eta, ttt_lr_eta, ln_weight, ln_bias, d_out, mini_batch,
                               eps, d_state_out, static_scratch, into, int(kernel_hint), saved)


@dataclass
class TTTMLPState:
    """mlp.rs:43-53: w1 [B,H,d,4d], b1 [B,H,4d], w2 [B,H,4d,d], b2 [B,H,d], always f32."""
    w1: torch.Tensor
    b1: torch.Tensor
    w2: torch.Tensor
    b2: torch.Tensor


class FusedMlp:
    """Fused TTT-MLP layer with the TTTMLP parameter set (mlp.rs:29-41) and the TTTInnerModel
    surface (inner.rs:13-58)."""

    def __init__(self, config: ModelConfig, w1_init, b1_init, w2_init, b2_init, ln_weight, ln_bias):
        H, d = config.num_heads, config.head_dim
        m = config.ttt.mlp_expansion_factor * d
        self.config = config
        self.w1_init = _need(w1_init, (H, d, m), torch.float32, "w1_init")
        self.b1_init = _need(b1_init, (H, m), torch.float32, "b1_init")
        self.w2_init = _need(w2_init, (H, m, d), torch.float32, "w2_init")
        self.b2_init = _need(b2_init, (H, d), torch.float32, "b2_init")
        self.ln_weight = _need(ln_weight, (H, d), torch.float32, "ln_weight")
        self.ln_bias = _need(ln_bias, (H, d), torch.float32, "ln_bias")

    @staticmethod
    def name() -> str:
        return "FusedTTTMLP"

    @classmethod
    def new(cls, config: ModelConfig, device, generator: Optional[torch.Generator] = None):
        """TTTMLP::new (mlp.rs:76-113): every parameter ~ Normal(0, 0.02)."""
        H, d = config.num_heads, config.head_dim
        m = config.ttt.mlp_expansion_factor * d

        def init(*shape):
            return (torch.randn(*shape, generator=generator, dtype=torch.float32) * 0.02).to(device)

        return cls(config, init(H, d, m), init(H, m), init(H, m, d), init(H, d), init(H, d), init(H, d))

    def get_config(self) -> ModelConfig:
        return self.config

    def init_state(self, batch_size: int) -> TTTMLPState:
        """mlp.rs:119-125."""
        rep = lambda p: p.unsqueeze(0).repeat(batch_size, *([1] * p.dim()))
        return TTTMLPState(rep(self.w1_init), rep(self.b1_init), rep(self.w2_init), rep(self.b2_init))

    def _launch(self, state: TTTMLPState, inputs: TTTInputsInner, mini_batch: int):
        out, state.w1, state.b1, state.w2, state.b2 = ttt_mlp_forward_raw(
            inputs.qkv.xq, inputs.qkv.xk, inputs.qkv.xv, state.w1, state.b1, state.w2, state.b2,
            inputs.token_eta, inputs.ttt_lr_eta, self.ln_weight, self.ln_bias, mini_batch,
            self.config.ttt.epsilon)
        return out

    def forward(self, state: TTTMLPState, inputs: TTTInputsInner) -> torch.Tensor:
        """inner.rs:25-50 in at most two launches: all full mini-batches, then the remainder."""
        K = self.config.ttt.mini_batch_size
        seq = inputs.qkv.xq.shape[2]
        full = (seq // K) * K
        outs = []
        if full > 0:
            outs.append(self._launch(state, inputs.slice_seq(range(0, full)), K))
        if full < seq:
            outs.append(self._launch(state, inputs.slice_seq(range(full, seq)), seq - full))
        return outs[0] if len(outs) == 1 else torch.cat(outs, 2)

    def forward_mini_batch(self, state: TTTMLPState, inputs: TTTInputsInner, r: range) -> torch.Tensor:
        if len(r) > self.config.ttt.mini_batch_size or len(r) == 0:
            raise _lib.TttError(_lib.TTT_ERR_SHAPE, "range longer than mini_batch_size")
        return self._launch(state, inputs.slice_seq(r), len(r))

    def backward(self, state0: Optional[TTTMLPState], inputs: TTTInputsInner, grad_output, grad_state_out=None):
        """Gradients of forward() over a sequence that is a multiple of mini_batch_size, starting from
        state0 (None: the [H,..] parameters broadcast over batch, init_state).  The reference gets these
        from Burn autodiff over mlp.rs:127-208.  Returns the dict of ttt_mlp_backward_raw."""
        st = (self.w1_init, self.b1_init, self.w2_init, self.b2_init) if state0 is None else \
            (state0.w1, state0.b1, state0.w2, state0.b2)
        return ttt_mlp_backward_raw(inputs.qkv.xq, inputs.qkv.xk, inputs.qkv.xv, *st, inputs.token_eta,
                                    inputs.ttt_lr_eta, self.ln_weight, self.ln_bias, grad_output,
                                    self.config.ttt.mini_batch_size, self.config.ttt.epsilon,
                                    d_state_out=grad_state_out)


class FusedTileMulti:
    """`fused-tile-multi` TTT-Linear layer: Fused<B, TTTLinear<B>, TileMultiKernel>.

    Holds the same parameters as TTTLinear (weight_init [H,d,d], bias_init [H,d], LayerNorm
    weight/bias [H,d]; linear.rs:17-25) so records are interchangeable with the plain layer
    (rust/fused/src/lib.rs:183-277).
    """

    def __init__(self, config: ModelConfig, weight_init, bias_init, ln_weight, ln_bias):
        H, d = config.num_heads, config.head_dim
        self.config = config
        self.weight_init = _need(weight_init, (H, d, d), torch.float32, "weight_init")
        self.bias_init = _need(bias_init, (H, d), torch.float32, "bias_init")
        self.ln_weight = _need(ln_weight, (H, d), torch.float32, "ln_weight")
        self.ln_bias = _need(ln_bias, (H, d), torch.float32, "ln_bias")

    @staticmethod
    def name() -> str:
        return "FusedTileMultiTTTLinear"  # wrapper.rs:85-87

    @classmethod
    def new(cls, config: ModelConfig, device, generator: Optional[torch.Generator] = None):
        """TTTLinear::new (linear.rs:54-78): every parameter ~ Normal(0, 0.02)."""
        H, d = config.num_heads, config.head_dim

        def init(*shape):
            return (torch.randn(*shape, generator=generator, dtype=torch.float32) * 0.02).to(device)

        return cls(config, init(H, d, d), init(H, d), init(H, d), init(H, d))

    def get_config(self) -> ModelConfig:
        return self.config

    def init_state(self, batch_size: int) -> TTTLinearState:
        """linear.rs:84-89: parameters repeated over the batch."""
        return TTTLinearState(self.weight_init.unsqueeze(0).repeat(batch_size, 1, 1, 1),
                              self.bias_init.unsqueeze(0).repeat(batch_size, 1, 1))

    def _pass(self, state: TTTLinearState, inputs: TTTInputsInner, start: int, stop: int):
        q, t = inputs.qkv, self.config.ttt
        out, state.weight, state.bias = host().linear_layer_forward(
            q.xq, q.xk, q.xv, state.weight, state.bias, inputs.token_eta, inputs.ttt_lr_eta, self.ln_weight,
            self.ln_bias, t.mini_batch_size, t.epsilon, t.checkpoint_interval, start, stop)
        return out

    def forward(self, state: TTTLinearState, inputs: TTTInputsInner) -> torch.Tensor:
        """wrapper.rs:102-164: all full mini-batches in one launch; a trailing remainder is one
        short mini-batch, as the Burn-op model does it (inner.rs:40-47), of the same launch where the library has one
        (ttt_linear_fwd_with_rest) and of a second one elsewhere.  Both launches read and write
        windows of the sequence in place.  A sequence without tokens leaves the state as it is."""
        seq = inputs.qkv.xq.shape[2]
        return self._pass(state, inputs, 0, seq) if seq > 0 else torch.empty_like(inputs.qkv.xq)

    def forward_mini_batch(self, state: TTTLinearState, inputs: TTTInputsInner, r: range) -> torch.Tensor:
        """wrapper.rs:166-211: one mini-batch (len(r) <= mini_batch_size)."""
        if len(r) > self.config.ttt.mini_batch_size or len(r) == 0:
            raise _lib.TttError(_lib.TTT_ERR_SHAPE, "range longer than mini_batch_size")
        return self._pass(state, inputs, r.start, r.stop)


@dataclass
class TTTLinearAdamState:
    """linear_adam.rs:28-44: state, first and second moments (per batch element, f32) and the step counter."""
    weight: torch.Tensor
    bias: torch.Tensor
    weight_m: torch.Tensor
    bias_m: torch.Tensor
    weight_v: torch.Tensor
    bias_v: torch.Tensor
    step: int = 0


@dataclass
class TTTLinearAdamConfig:
    """linear_adam.rs:46-62."""
    beta1: float = 0.9
    beta2: float = 0.999
    epsilon: float = 1e-8
    lr: float = 1e-3


class FusedLinearAdam:
    """TTTLinearAdam (rust/core/src/linear_adam.rs) on the fused kernel: the parameters of TTTLinear, an Adam step
    on the eta-weighted gradients per mini-batch instead of the plain update."""

    def __init__(self, config: ModelConfig, adam: TTTLinearAdamConfig, weight_init, bias_init, ln_weight, ln_bias):
        H, d = config.num_heads, config.head_dim
        self.config, self.adam = config, adam
        self.weight_init = _need(weight_init, (H, d, d), torch.float32, "weight_init")
        self.bias_init = _need(bias_init, (H, d), torch.float32, "bias_init")
        self.ln_weight = _need(ln_weight, (H, d), torch.float32, "ln_weight")
        self.ln_bias = _need(ln_bias, (H, d), torch.float32, "ln_bias")

    @staticmethod
    def name() -> str:
        return "TTTLinearAdam"  # linear_adam.rs:134-136

    def get_config(self) -> ModelConfig:
        return self.config

    def init_state(self, batch_size: int) -> TTTLinearAdamState:
        """linear_adam.rs:164-177: parameters repeated over the batch, zero moments, step 0."""
        w = self.weight_init.unsqueeze(0).repeat(batch_size, 1, 1, 1)
        b = self.bias_init.unsqueeze(0).repeat(batch_size, 1, 1)
        return TTTLinearAdamState(w, b, torch.zeros_like(w), torch.zeros_like(b), torch.zeros_like(w),
                                  torch.zeros_like(b), 0)

    def _launch(self, state: TTTLinearAdamState, inputs: TTTInputsInner, mini_batch: int):
        a = self.adam
        out, w, b, mo, step = ttt_linear_adam_forward_raw(
            inputs.qkv.xq, inputs.qkv.xk, inputs.qkv.xv, state.weight, state.bias, inputs.token_eta,
            inputs.ttt_lr_eta, self.ln_weight, self.ln_bias, mini_batch, a.beta1, a.beta2, a.epsilon, a.lr,
            moments=(state.weight_m, state.bias_m, state.weight_v, state.bias_v), step=state.step,
            eps=self.config.ttt.epsilon)
        state.weight, state.bias = w, b
        state.weight_m, state.bias_m, state.weight_v, state.bias_v = mo
        state.step = step
        return out

    def forward(self, state: TTTLinearAdamState, inputs: TTTInputsInner) -> torch.Tensor:
        """inner.rs:25-50: all full mini-batches in one launch, a trailing remainder as one short mini-batch."""
        K = self.config.ttt.mini_batch_size
        seq = inputs.qkv.xq.shape[2]
        full = (seq // K) * K
        outs = []
        if full > 0:
            outs.append(self._launch(state, inputs.slice_seq(range(0, full)), K))
        if full < seq:
            outs.append(self._launch(state, inputs.slice_seq(range(full, seq)), seq - full))
        return outs[0] if len(outs) == 1 else torch.cat(outs, 2)

    def forward_mini_batch(self, state: TTTLinearAdamState, inputs: TTTInputsInner, r: range) -> torch.Tensor:
        if len(r) > self.config.ttt.mini_batch_size or len(r) == 0:
            raise _lib.TttError(_lib.TTT_ERR_SHAPE, "range longer than mini_batch_size")
        return self._launch(state, inputs.slice_seq(r), len(r))


@dataclass
class TTTMLPNState:
    """mlp2.rs:38-53, mlp3.rs:42-53, mlp4.rs:46-59: the n_hidden + 1 weight layers [B,H,in,out] and biases [B,H,out],
    always f32."""
    weights: list
    biases: list


class FusedMlpN:
    """TTTMLP2 / TTTMLP3 / TTTMLP4 (rust/core/src/mlp2.rs, mlp3.rs, mlp4.rs) on the fused kernel: d -> 4d -> ... -> 4d
    -> d with 2, 3 or 4 hidden layers, the TTTInnerModel interface of rust/core/src/inner.rs:13-58.  kernel_hint: that of
    ttt_mlpn_forward_raw, for every call."""

    def __init__(self, config: ModelConfig, weights_init, biases_init, ln_weight, ln_bias, kernel_hint: int = 0):
        H, d = config.num_heads, config.head_dim
        n = len(weights_init) - 1
        if n < 2 or n > 4 or len(biases_init) != n + 1:
            raise _lib.TttError(_lib.TTT_ERR_UNSUPPORTED, "FusedMlpN: 2, 3 or 4 hidden layers")
        dims = [d] + [4 * d] * n + [d]
        self.config, self.n_hidden, self.kernel_hint = config, n, kernel_hint
        self.weights_init = [_need(w, (H, dims[i], dims[i + 1]), torch.float32, f"weights_init[{i}]")
                             for i, w in enumerate(weights_init)]
        self.biases_init = [_need(b, (H, dims[i + 1]), torch.float32, f"biases_init[{i}]")
                            for i, b in enumerate(biases_init)]
        self.ln_weight = _need(ln_weight, (H, d), torch.float32, "ln_weight")
        self.ln_bias = _need(ln_bias, (H, d), torch.float32, "ln_bias")

    def name(self) -> str:
        return f"TTTMLP{self.n_hidden}"  # mlp2.rs:70-72, mlp3.rs:70-72, mlp4.rs:76-78

    def get_config(self) -> ModelConfig:
        return self.config

    def init_state(self, batch_size: int) -> TTTMLPNState:
        """mlp2.rs:129-145 and its siblings: the parameters repeated over the batch."""
        rep = lambda t: t.unsqueeze(0).repeat(batch_size, *([1] * t.dim()))
        return TTTMLPNState([rep(w) for w in self.weights_init], [rep(b) for b in self.biases_init])

    def _launch(self, state: TTTMLPNState, inputs: TTTInputsInner, mini_batch: int):
        out, ws, bs = ttt_mlpn_forward_raw(inputs.qkv.xq, inputs.qkv.xk, inputs.qkv.xv, state.weights, state.biases,
                                           inputs.token_eta, inputs.ttt_lr_eta, self.ln_weight, self.ln_bias,
                                           mini_batch, self.config.ttt.epsilon, self.kernel_hint)
        state.weights, state.biases = ws, bs
        return out

    def forward(self, state: TTTMLPNState, inputs: TTTInputsInner) -> torch.Tensor:
        """inner.rs:25-50: all full mini-batches in one launch, a trailing remainder as one short mini-batch."""
        K = self.config.ttt.mini_batch_size
        seq = inputs.qkv.xq.shape[2]
        full = (seq // K) * K
        outs = []
        if full > 0:
            outs.append(self._launch(state, inputs.slice_seq(range(0, full)), K))
        if full < seq:
            outs.append(self._launch(state, inputs.slice_seq(range(full, seq)), seq - full))
        return outs[0] if len(outs) == 1 else torch.cat(outs, 2)

    def forward_mini_batch(self, state: TTTMLPNState, inputs: TTTInputsInner, r: range) -> torch.Tensor:
        if len(r) > self.config.ttt.mini_batch_size or len(r) == 0:
            raise _lib.TttError(_lib.TTT_ERR_SHAPE, "range longer than mini_batch_size")
        return self._launch(state, inputs.slice_seq(r), len(r))


def ttt_stack_workspace_bytes(B: int, H: int, seq: int, d: int, mini_batch: int, io: torch.dtype, mlp_flags,
                              chunk_tokens: int = 0) -> int:
    """ttt_stack_fwd_workspace_bytes for a stack whose layer l is TTT-MLP where mlp_flags[l] is true."""
    desc = TttDesc(B, H, seq, d, mini_batch, 1e-6, 1, _lib.TTT_BF16 if io == torch.bfloat16 else _lib.TTT_F32)
    arr = (_lib.TttStackLayer * len(mlp_flags))()
    for a, f in zip(arr, mlp_flags):
        a.kind = 1 if f else 0
    n = lib().ttt_stack_fwd_workspace_bytes(C.byref(desc), len(mlp_flags), arr, chunk_tokens)
    if n < 0:
        raise _lib.TttError(_lib.TTT_ERR_SHAPE, lib().ttt_last_error().decode())
    return n


def mlp_fwd_lost_workgroups() -> int:
    """ttt_mlp_fwd_lost_workgroups of the current device: how many workgroups of the kernels that put a unit on two of them
    (TTT-MLP forward at head_dim 128 with bf16 I/O, TTT-MLP backward, TTT-Linear backward with f32 I/O, TTT-MLP with several hidden
    layers) gave up waiting for their partner since the library was loaded.  The unit's results are then NaN as those calls
    say; ttt_mlpn_forward_raw's are right all the same.  A blocking copy from the device; meaningful once the work in
    question has finished."""
    n = C.c_int64(0)
    check(lib().ttt_mlp_fwd_lost_workgroups(C.byref(n)))
    return n.value


def ttt_stack_forward_raw(layers, token_eta, mini_batch: int, eps: float = 1e-6, kernel_hint: int = 0,
                          workspace: Optional[torch.Tensor] = None, chunk_tokens: int = 0,
                          aux_stream: Optional[torch.cuda.Stream] = None, check_lost: Optional[bool] = None):
    """One call of ttt_stack_fwd on the current stream: inner models applied layer by layer, layer l on
    xq = x + pq, xk = x + pk, xv = x + pv with x the previous layer's output (0 for the first layer).
    chunk_tokens > 0 runs the layers as a wavefront over sequence windows of that many tokens (layer l + 1 works on
    a window as soon as layer l has left it; windows that are ready together share a launch); aux_stream, a second
    torch.cuda.Stream, lets the TTT-MLP launches run beside the TTT-Linear ones.
    layers: list of dicts with pq, pk, pv [B,H,seq,d], lr [B,H,seq], gamma, beta [H,d] and either W0, b0
    (TTT-Linear) or W1, b1, W2, b2 (TTT-MLP), parameters [H,..].  Returns (out, states) with states[l] the final
    state tensors of layer l (per batch element).
    check_lost: a stack with a TTT-MLP layer at head_dim 128 and bf16 I/O runs the two-CU kernel, whose failure
    (a workgroup that waited for its partner in vain) shows only in the data (NaN) and in the device's status word.
    With check_lost the call waits for the device, reads that word before and after and raises if it moved.
    Default (None): checked unless the current stream is being captured into a graph; callers that must not
    synchronise (timed loops) pass False and compare mlp_fwd_lost_workgroups() around their own region."""
    if check_lost is None:
        check_lost = not torch.cuda.is_current_stream_capturing()
    # aux_stream reads and writes tensors that torch's allocator ties to the current stream only; the call joins
    # it into the current stream before it returns, so later work on that stream is ordered after it
    return host().stack_forward(layers, token_eta, mini_batch, eps, kernel_hint, workspace, chunk_tokens,
                                0 if aux_stream is None else aux_stream.cuda_stream, int(check_lost))


# --------------------------------------------------------------------------- either side of the inner loop
def rope_cos_sin(seq_len: int, offset: int, wrap: Optional[int], head_dim: int, device, base: float = 10000.0):
    """RotaryEmbeddingConfig::init + RotaryEmbedding::get_cos_sin (rust/core/src/util.rs:266-322) in f32:
    returns (cos, sin) [seq_len, head_dim/2] (the reference repeats this half twice)."""
    half = head_dim // 2
    inv_freq = torch.tensor([1.0 / base ** ((2 * i) / head_dim) for i in range(half)], dtype=torch.float32)
    pos = torch.arange(seq_len, dtype=torch.float32) + float(offset)
    if wrap is not None:
        pos = torch.remainder(pos, float(wrap))
    freqs = pos[:, None] * inv_freq[None, :]
    return freqs.cos().to(device), freqs.sin().to(device)


def ttt_lr_eta_logit_grad(grad_ttt_lr_eta, lr_logits, base_lr: float, head_dim: int):
    """Gradient w.r.t. the lr-gate logits from grad_ttt_lr_eta (an output of ttt_linear_backward_raw /
    ttt_mlp_backward_raw): the chain through ttt_lr_eta = base_lr * sigmoid(logit) / head_dim (get_lr,
    rust/layer/src/ttt.rs:205-227).  The reference leaves this step to Burn autodiff outside the fused kernel's
    boundary; here it is one elementwise expression on the caller's device, in f32."""
    s = torch.sigmoid(lr_logits.float())
    return grad_ttt_lr_eta.float() * (base_lr / head_dim) * s * (1.0 - s)


def inner_loop_inputs_raw(xq, xk, xv, lr_logits, lr_bias, base_lr: float, token_idx, learnable_token_idx,
                          mini_batch: int, rope=None, pos_offset: int = 0, pos_wrap: int = 0) -> TTTInputsInner:
    """One call of ttt_inner_inputs: TTT::get_inner_loop_inputs after the projections
    (rust/layer/src/ttt.rs:147-194, 205-227, 247-268).  xq,xk,xv [B,seq,H,d]; lr_logits [B,seq,H];
    rope = (cos, sin) tables [npos, d/2] f32 or None."""
    cos, sin = (None, None) if rope is None else rope
    q, k, v, lr, te = host().inner_inputs(xq, xk, xv, lr_logits, lr_bias, token_idx, learnable_token_idx, cos, sin,
                                          pos_offset, pos_wrap, mini_batch, base_lr)
    return TTTInputsInner(Qkv(q, k, v), te, lr)


def ttt_linear_forward_fused_inputs_raw(xq, xk, xv, lr_logits, lr_bias, base_lr: float, token_idx,
                                        learnable_token_idx, weight, bias, ln_weight, ln_bias, mini_batch: int,
                                        rope=None, pos_offset: int = 0, pos_wrap: int = 0, eps: float = 1e-6,
                                        checkpoint_interval: int = 1, want_checkpoints: bool = False,
                                        packed_checkpoints: int = 0, save_inputs: bool = False):
    """One call of ttt_linear_fwd_fused_inputs: inner_loop_inputs_raw and ttt_linear_forward_raw in one kernel
    (rust/layer/src/ttt.rs:147-268 followed by rust/kernels/src/kernel.rs:62-69).  xq,xk,xv [B,seq,H,d];
    lr_logits [B,seq,H]; rope = (cos, sin) tables [npos, d/2] f32 or None; weight/bias/ln_* as for
    ttt_linear_forward_raw.  Returns (output, weight_out, bias_out[, weight_ckpt, bias_ckpt][, TTTInputsInner]):
    the last item, with save_inputs, holds the operands as the kernel used them (what the backward needs)."""
    cos, sin = (None, None) if rope is None else rope
    r = host().linear_forward_fused_inputs(xq, xk, xv, lr_logits, lr_bias, token_idx, learnable_token_idx, cos, sin,
                                           pos_offset, pos_wrap, mini_batch, base_lr, weight, bias, ln_weight, ln_bias,
                                           eps, checkpoint_interval, want_checkpoints, int(packed_checkpoints),
                                           save_inputs)
    if not save_inputs:
        return r
    q, k, v, lr, te = r[-5:]
    return r[:-5] + (TTTInputsInner(Qkv(q, k, v), te, lr),)


def layer_epilogue_raw(inner_out, post_norm_weight, post_norm_bias, gate=None, eps: float = 1e-6):
    """One call of ttt_layer_epilogue: head merge + post_norm LayerNorm (+ tanh-GELU gate) of
    TTT::forward (rust/layer/src/ttt.rs:285-297).  inner_out [B,H,seq,d] -> [B,seq,H*d]."""
    return host().layer_epilogue(inner_out, post_norm_weight, post_norm_bias, gate, eps)
