"""A KDA layer composed from this backend's kernels.

The caller path of the operators in the reference is
``KimiDeltaAttention.forward`` (src/kda/kda.py:98-206): the projections
(src/kda/projections.py:144-225), the lower-bounded decay (src/kda/decay.py:28-43),
the operator (``recurrent_kda`` for ``mode="recurrent"``/``"decode"``,
``chunkwise_kda`` otherwise, kda.py:133-151), the head-wise RMSNorm and the
output gate (kda.py:153-161) and the ``KDAState`` handed to the next call
(kda.py:163-183).  ``kda_attention_forward`` runs that path on the GPU:

* q, k, v: the projection GEMM (``torch.nn.functional.linear``, as the
  reference's ``nn.Linear``), then ``fused.conv_silu`` (ShortConv + SiLU, L2
  norm per head for q and k, right padding and the decode history);
* beta and the decay: their projections, then ``fused.layer_gates``, which
  feeds the operator (the chunk kernel can also form g from the logits
  itself, ``fused.chunkwise_kda_with_decay``, bit-identical but measured
  slower, so the layer runs two launches);
* output: ``fused.rmsnorm_gate`` (RMSNorm times the sigmoid gate of the gate
  projection), the output projection, and the mask.

The projection GEMMs are torch's; everything between them runs in this
library's HIP kernels.  A decode step of up to ``DECODE_STEP_BATCH`` sequences
outside autograd runs projections and all in three launches
(``kda_layer_decode``), with the same roundings between the stages.  Weights are plain tensors (``KDALayerWeights``), so a
reference module's parameters can be handed over with ``from_module``.
"""

from __future__ import annotations

import ctypes
from dataclasses import dataclass
from typing import Literal

import torch
import torch.nn.functional as F

from . import _lib, _prep, fused
from .chunkwise import checked_chunkwise
from .recurrent import checked_recurrent
from .state import KDAState, ShortConvState
from .utils import checked_lengths, validate_core_inputs


@dataclass
class KDALayerWeights:
    """The parameters of one KDA layer, in the reference's layouts
    (src/kda/projections.py:35-73, src/kda/decay.py:24-26, src/kda/kda.py:50-62):
    linear weights ``[out, in]``, ShortConv weights ``[C, K_conv]`` in lag order."""

    num_heads: int
    key_head_dim: int
    value_head_dim: int
    q_proj: torch.Tensor
    k_proj: torch.Tensor
    v_proj: torch.Tensor
    q_conv: torch.Tensor
    k_conv: torch.Tensor
    v_conv: torch.Tensor
    beta_proj: torch.Tensor
    alpha_down: torch.Tensor
    alpha_up: torch.Tensor
    b_alpha: torch.Tensor
    a_log: torch.Tensor
    norm_weight: torch.Tensor | None
    gate_proj: torch.Tensor
    output_proj: torch.Tensor
    g_min: float = -5.0
    eps: float = 1e-6
    accumulate_state_in_fp32: bool = True
    q_proj_bias: torch.Tensor | None = None
    k_proj_bias: torch.Tensor | None = None
    v_proj_bias: torch.Tensor | None = None
    q_conv_bias: torch.Tensor | None = None
    k_conv_bias: torch.Tensor | None = None
    v_conv_bias: torch.Tensor | None = None
    beta_bias: torch.Tensor | None = None
    gate_bias: torch.Tensor | None = None
    output_bias: torch.Tensor | None = None

    @property
    def d_model(self) -> int:
        return self.gate_proj.shape[0]

    @property
    def key_width(self) -> int:
        return self.num_heads * self.key_head_dim

    @property
    def value_width(self) -> int:
        return self.num_heads * self.value_head_dim

    @property
    def conv_kernel_size(self) -> int:
        return self.q_conv.shape[1]

    @classmethod
    def from_module(cls, module, *, detach: bool = True) -> "KDALayerWeights":
        """The parameters of a module with the reference's attribute names
        (``KimiDeltaAttention``, src/kda/kda.py:45-62).  ``detach=False``
        keeps the module's parameters themselves, so that a backward through
        ``kda_attention_forward`` fills their ``.grad`` (training);
        the default hands over detached views (inference)."""
        cfg, p = module.config, module.projections
        d = (lambda t: t.detach()) if detach else (lambda t: t)  # noqa: E731
        bias = lambda lin: None if lin.bias is None else d(lin.bias)  # noqa: E731
        conv_bias = lambda c: None if c.bias is None else d(c.bias)  # noqa: E731
        norm = module.output_norm.weight
        return cls(
            num_heads=cfg.num_heads, key_head_dim=cfg.key_head_dim, value_head_dim=cfg.value_head_dim,
            q_proj=d(p.q_proj.weight), k_proj=d(p.k_proj.weight), v_proj=d(p.v_proj.weight),
            q_conv=d(p.q_conv.weight), k_conv=d(p.k_conv.weight), v_conv=d(p.v_conv.weight),
            beta_proj=d(p.beta_proj.weight), alpha_down=d(p.alpha_down.weight),
            alpha_up=d(p.alpha_up.weight), b_alpha=d(p.b_alpha), a_log=d(module.decay.A_log),
            norm_weight=None if norm is None else d(norm),
            gate_proj=d(module.output_gate.gate_proj.weight),
            output_proj=d(module.output_gate.output_proj.weight),
            g_min=cfg.g_min, eps=cfg.eps, accumulate_state_in_fp32=cfg.accumulate_state_in_fp32,
            q_proj_bias=bias(p.q_proj), k_proj_bias=bias(p.k_proj), v_proj_bias=bias(p.v_proj),
            q_conv_bias=conv_bias(p.q_conv), k_conv_bias=conv_bias(p.k_conv), v_conv_bias=conv_bias(p.v_conv),
            beta_bias=bias(p.beta_proj), gate_bias=bias(module.output_gate.gate_proj),
            output_bias=bias(module.output_gate.output_proj),
        )


@dataclass
class KDALayerOutput:
    """Output and next cache state of one layer call (src/kda/kda.py:29-35)."""

    hidden_states: torch.Tensor
    state: KDAState | None = None


def _validate_state(w: KDALayerWeights, hidden_states: torch.Tensor, state: KDAState | None) -> None:
    """The cache-shape checks of KimiDeltaAttention._validate_state (src/kda/kda.py:64-96)."""
    if state is None:
        return
    batch = hidden_states.shape[0]
    expected_recurrent = (batch, w.num_heads, w.key_head_dim, w.value_head_dim)
    if state.recurrent_state.shape != expected_recurrent:
        raise ValueError(f"state recurrent tensor must have shape {expected_recurrent}")
    history = w.conv_kernel_size - 1
    expected_buffers = ((batch, history, w.key_width), (batch, history, w.key_width), (batch, history, w.value_width))
    actual_buffers = (state.q_conv_state.buffer.shape, state.k_conv_state.buffer.shape,
                      state.v_conv_state.buffer.shape)
    if actual_buffers != expected_buffers:
        raise ValueError(f"state ShortConv buffers must have shapes {expected_buffers}")
    if state.recurrent_state.device != hidden_states.device:
        raise ValueError("state and hidden_states must be on the same device")


# The calls the native decode step takes: up to DECODE_STEP_BATCH sequences whose
# projections take at most DECODE_STEP_PRODUCTS multiply-adds.  Its projections
# read the weights again for every 64 sequences, while the composed stages are
# bound by the host at about 240 us a call until their GEMMs take longer than
# that.  Measured per call (us, heads x 128 = d_model, bf16), native against
# composed:
#   d_model 2048: 4 sequences 37 / 238, 32 49 / 239, 128 127 / 239, 256 228 / 242;
#   d_model 4096: 32 98 / 238, 65 (5.5e9 products) 201 / 239, 128 (1.1e10) 297 / 258,
#     256 557 / 348;
#   d_model 7168: 4 134 / 239, 32 (8.3e9) 258 / 254, 64 (1.7e10) 417 / 303.
# A captured call has no host time: its line is where the device times meet, at
# 128-wide heads (with key or value heads of 64 the composed stages' device time
# is the longer one up to DECODE_STEP_PRODUCTS: 1.2 to 2.9 times).  There, replays
# of the two, native over composed:
#   d_model 1024: 256 sequences 0.91;  1536: 160 0.94, 192 1.03;
#   2048: 128 0.88, 192 (3.9e5 activations) 1.06, 256 1.16;  2560: 64 0.83, 128 1.01;
#   3072: 64 0.83, 96 (2.9e5) 1.09;  4096: 48 0.95, 64 (5.4e9 products) 1.01, 96 1.11;
#   5120: 32 0.94, 64 1.22;  6144: 24 0.95, 48 1.12;  7168: 16 0.98, 24 (6.2e9) 1.07.
DECODE_STEP_BATCH = 256
DECODE_STEP_PRODUCTS = 8_000_000_000
CAPTURED_STEP_PRODUCTS = 5_000_000_000
CAPTURED_STEP_ACTIVATIONS = 1 << 18


def _products(w: KDALayerWeights, batch: int) -> int:
    """Multiply-adds of the token's projections."""
    weights = (w.q_proj, w.k_proj, w.v_proj, w.beta_proj, w.alpha_down, w.alpha_up, w.gate_proj, w.output_proj)
    return batch * sum(t.numel() for t in weights)


def _few_products(w: KDALayerWeights, batch: int) -> bool:
    """Whether the token's projections keep to DECODE_STEP_PRODUCTS."""
    return _products(w, batch) <= DECODE_STEP_PRODUCTS


def _captured_past_the_line(w: KDALayerWeights, batch: int) -> bool:
    """Whether the call is being captured into a graph and its replays take
    longer in the native step than in the composed stages."""
    if w.key_head_dim != 128 or w.value_head_dim != 128 or not torch.cuda.is_current_stream_capturing():
        return False
    return batch * w.q_proj.shape[1] > CAPTURED_STEP_ACTIVATIONS or _products(w, batch) > CAPTURED_STEP_PRODUCTS


_PLAIN = (torch.Tensor, torch.nn.Parameter)


def _transformed() -> bool:
    """Whether a torch.func transform or a forward-mode level is active: its
    tensors look like plain ones, and torch's own stages (the projections) take
    them where a native call does not see them."""
    return torch._C._functorch.peek_interpreter_stack() is not None or torch.autograd.forward_ad._current_level >= 0


def _decode_step(w: KDALayerWeights, x: torch.Tensor, state: KDAState | None, in_place: bool) -> KDALayerOutput | None:
    """One token per sequence through ``kda_layer_decode``, or None when the call
    needs the composed stages: tensors that require grad, autocast, torch.func
    transforms, tensor subclasses, layouts, dtypes or sizes the kernels do not take, or anything
    the stages would refuse (so that they raise their own errors)."""
    batch, H, K, V = x.shape[0], w.num_heads, w.key_head_dim, w.value_head_dim
    dtype, device = x.dtype, x.device
    if (batch > DECODE_STEP_BATCH or dtype not in (torch.bfloat16, torch.float16) or device.type != "cuda"
            or K not in (64, 128) or V not in (64, 128) or not w.accumulate_state_in_fp32
            or torch.is_autocast_enabled("cuda") or _transformed() or not w.eps > 0 or not w.g_min < 0):
        return None
    if not batch:
        return None
    for t in (w.q_proj, w.k_proj, w.v_proj, w.beta_proj, w.alpha_down, w.alpha_up, w.gate_proj, w.output_proj,
              w.q_conv, w.k_conv, w.v_conv, w.b_alpha, w.a_log):
        if t is None:  # the stages take a layer without a decay bias, and refuse the rest
            return None
    if w.q_conv.ndim != 2 or w.q_proj.ndim != 2 or w.alpha_down.ndim != 2 or w.output_proj.ndim != 2:
        return None
    if not _few_products(w, batch) or _captured_past_the_line(w, batch):
        return None
    d_model, kw, vw, taps = x.shape[2], H * K, H * V, w.q_conv.shape[1]
    rank, out_dim = w.alpha_down.shape[0], w.output_proj.shape[0]
    norm = w.norm_weight
    per_head = norm is not None and norm.ndim == 2
    if (d_model % 64 or d_model != vw or not 1 <= taps <= 8 or rank % 8 or not 8 <= rank <= 256
            or w.a_log.dtype != torch.float32):
        return None
    hist = (batch, taps - 1)
    expected = [
        (x, (batch, 1, d_model)), (w.q_proj, (kw, d_model)), (w.k_proj, (kw, d_model)), (w.v_proj, (vw, d_model)),
        (w.beta_proj, (H, d_model)), (w.alpha_down, (rank, d_model)), (w.gate_proj, (vw, d_model)),
        (w.alpha_up, (kw, rank)), (w.output_proj, (out_dim, vw)), (w.q_proj_bias, (kw,)), (w.k_proj_bias, (kw,)),
        (w.v_proj_bias, (vw,)), (w.beta_bias, (H,)), (w.gate_bias, (vw,)), (w.output_bias, (out_dim,)),
        (w.q_conv, (kw, taps)), (w.k_conv, (kw, taps)), (w.v_conv, (vw, taps)), (w.q_conv_bias, (kw,)),
        (w.k_conv_bias, (kw,)), (w.v_conv_bias, (vw,)), (w.b_alpha, (H, K)), (w.a_log, (H,)),
        (norm, (H, V) if per_head else (V,)),
    ]
    buffers = (None, None, None)
    recurrent = offset = None
    if state is not None:
        recurrent, offset = state.recurrent_state, state.sequence_offset
        if recurrent.dtype != torch.float32 or offset.device != device:
            return None
        buffers = (state.q_conv_state.buffer, state.k_conv_state.buffer, state.v_conv_state.buffer)
        expected += [(buffers[0], (*hist, kw)), (buffers[1], (*hist, kw)), (buffers[2], (*hist, vw)),
                     (recurrent, (batch, H, K, V)), (offset, (batch,))]
    grad = torch.is_grad_enabled()
    for t, shape in expected:
        if t is not None and (
                type(t) not in _PLAIN or t.shape != shape or t.device != device or not t.is_contiguous()
                or (grad and t.requires_grad)
                or (t.dtype != dtype and t is not w.a_log and t is not recurrent and t is not offset)):
            return None
    ptr = [None if t is None else t.data_ptr() for t, _ in expected] + [None] * (29 - len(expected))
    if any(p is not None and p & 15 for p in (*ptr[:9], ptr[27])):
        return None
    lib = _lib.load()
    new = x.new_empty
    outs = [new(*hist, kw), new(*hist, kw), new(*hist, vw)]
    state_out = recurrent if in_place and recurrent is not None else new(batch, H, K, V, dtype=torch.float32)
    offset_out = new(batch, dtype=torch.long)
    out = new(batch, 1, out_dim)
    args = _lib.LayerDecodeArgs(
        *ptr, *(t.data_ptr() for t in outs), state_out.data_ptr(), offset_out.data_ptr(), out.data_ptr(), None, 0,
        batch, d_model, out_dim, H, K, V, taps, rank, float(w.g_min), float(w.eps), _lib.dtype_code(dtype),
        1 if per_head else 0)
    ref = ctypes.addressof(args)
    args.workspace_bytes = lib.kda_layer_decode_workspace_bytes(ref)
    workspace = _prep.workspace(args.workspace_bytes, device, "kda_attention_forward's decode step")
    args.workspace = workspace.data_ptr()
    _lib.check(lib.kda_layer_decode(ref, _prep.stream(device)))
    return KDALayerOutput(hidden_states=out, state=KDAState(
        recurrent_state=state_out, q_conv_state=ShortConvState(outs[0]), k_conv_state=ShortConvState(outs[1]),
        v_conv_state=ShortConvState(outs[2]), sequence_offset=offset_out))


def kda_attention_forward(
    w: KDALayerWeights,
    hidden_states: torch.Tensor,
    attention_mask: torch.Tensor | None = None,
    state: KDAState | None = None,
    mode: Literal["recurrent", "chunkwise", "decode"] = "chunkwise",
    output_final_state: bool = False,
    *,
    update_state_in_place: bool = False,
) -> KDALayerOutput:
    """One KDA layer call, as ``KimiDeltaAttention.forward`` (src/kda/kda.py:98-183)
    without the diagnostics.  ``update_state_in_place`` (decode only) writes the
    new recurrent state over ``state.recurrent_state`` instead of a new tensor."""
    if hidden_states.ndim != 3 or hidden_states.shape[-1] != w.d_model:
        raise ValueError(f"hidden_states must have shape [B,T,{w.d_model}], got {tuple(hidden_states.shape)}")
    batch, tokens, _ = hidden_states.shape
    if tokens == 0:
        raise ValueError("KDA does not support empty sequences")
    if mode not in ("recurrent", "chunkwise", "decode"):
        raise ValueError(f"unsupported KDA mode {mode!r}")
    if mode == "decode" and tokens != 1:
        raise ValueError("decode mode requires exactly one token")
    valid = checked_lengths(attention_mask, batch, tokens, hidden_states.device)
    _validate_state(w, hidden_states, state)
    x = hidden_states
    if mode == "decode" and attention_mask is None:
        step = _decode_step(w, x, state, update_state_in_place)
        if step is not None:
            return step
    H, K, V = w.num_heads, w.key_head_dim, w.value_head_dim
    return_state = output_final_state or mode == "decode"

    # projections (src/kda/projections.py:164-218)
    qs, ks, vs = (None, None, None) if state is None else (state.q_conv_state, state.k_conv_state,
                                                             state.v_conv_state)
    conv = fused.conv_silu_with_lengths
    q, q_next = conv(F.linear(x, w.q_proj, w.q_proj_bias), w.q_conv, w.q_conv_bias, qs, valid, num_heads=H,
                     normalize=True, eps=w.eps, output_final_state=return_state)
    k, k_next = conv(F.linear(x, w.k_proj, w.k_proj_bias), w.k_conv, w.k_conv_bias, ks, valid, num_heads=H,
                     normalize=True, eps=w.eps, output_final_state=return_state)
    v, v_next = conv(F.linear(x, w.v_proj, w.v_proj_bias), w.v_conv, w.v_conv_bias, vs, valid, num_heads=H,
                     normalize=False, eps=1e-6, output_final_state=return_state)
    beta_logits = F.linear(x, w.beta_proj, w.beta_bias)
    decay_logits = F.linear(F.linear(x, w.alpha_down), w.alpha_up).reshape(batch, tokens, H, K)

    # the operator (src/kda/kda.py:131-151)
    initial = None if state is None else state.recurrent_state
    keep_state = return_state
    # the decay kernel, then the operator: measured faster than forming g
    # inside the chunk kernel (fused.chunkwise_kda_with_decay, bit-identical),
    # whose extra VALU work lands on the chunk kernel's latency-bound loaders
    g, beta = fused.layer_gates(decay_logits, w.a_log, w.g_min, w.b_alpha, beta_logits)
    validate_core_inputs(q, k, v, g, beta, initial, None)
    if mode == "chunkwise":
        core = checked_chunkwise(q, k, v, g, beta, initial, keep_state, attention_mask, valid,
                                 w.accumulate_state_in_fp32)
    else:
        core = checked_recurrent(q, k, v, g, beta, initial, keep_state, attention_mask, valid,
                                 w.accumulate_state_in_fp32, update_state_in_place=update_state_in_place
                                 and mode == "decode" and initial is not None)

    # RMSNorm x output gate, output projection, mask (src/kda/kda.py:153-161)
    gated = fused.rmsnorm_gate(core.hidden_states, w.norm_weight, w.eps,
                               gate_logits=F.linear(x, w.gate_proj, w.gate_bias))
    out = F.linear(gated.reshape(batch, tokens, H * V), w.output_proj, w.output_bias)
    if attention_mask is not None:
        out = out * attention_mask[..., None].to(out.dtype)

    next_state = None
    if return_state:
        # src/kda/kda.py:163-183
        if valid is not None:
            offset = valid.to(torch.long) if state is None else state.sequence_offset.to(x.device) + valid
        elif state is None:
            offset = torch.full((batch,), tokens, dtype=torch.long, device=x.device)
        else:
            offset = state.sequence_offset.to(x.device) + tokens
        next_state = KDAState(recurrent_state=core.final_state, q_conv_state=q_next, k_conv_state=k_next,
                              v_conv_state=v_next, sequence_offset=offset)
    return KDALayerOutput(hidden_states=out, state=next_state)


__all__ = ["KDALayerOutput", "KDALayerWeights", "kda_attention_forward"]
