"""The calls a user of this framework makes, as measurable cases.

Kinds (each through the package's public entry points):

* ``decode``: ``recurrent_kda`` on one new token per sequence (a few tokens
  when a speculative draft is verified), the state updated functionally (the
  default) or in place (a serving loop's choice).
* ``prefill``: ``chunkwise_kda`` over whole prompts, dense, right-padded
  (``attention_mask``) or packed documents (``cu_seqlens``).
* ``train``: ``chunkwise_kda`` forward and backward, every input's gradient.
* ``layer``: ``layer.kda_attention_forward``, in decode, prefill (state
  returned) and training (forward + backward, every weight's gradient) use.
* ``cache``: ``cache.reorder_states`` over the decode caches of a model's
  layers (beam search's reorder).

Decays follow the layer's own gate, g = -5 sigmoid(.): a spread over the key
channels from slow (about -0.005 a token) to fast (about -2.5).  q and k are
L2-normalised per head as the layer hands them over, beta is a sigmoid.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch
import torch.nn.functional as F

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "kimi-k3-pytorch_amd"))

import kda  # noqa: E402
from kda.cache import reorder_states  # noqa: E402
from kda.layer import KDALayerWeights, kda_attention_forward  # noqa: E402
from kda.state import KDAState, ShortConvState  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
CONV = 4  # ShortConv taps of every layer (the reference's default)
STATE_STD = 0.02


def listed():
    return [
        # one user's next token: launch and host latency
        {"name": "decode_one", "kind": "decode", "dtype": "bf16", "batch": 1, "tokens": 1, "heads": 32, "key_dim": 128,
         "value_dim": 128, "in_place": False},
        # a full serving batch's next token, state updated in place
        {"name": "decode_batch", "kind": "decode", "dtype": "bf16", "batch": 256, "tokens": 1, "heads": 32,
         "key_dim": 128, "value_dim": 128, "in_place": True},
        # a whole layer's next token for a moderate batch
        {"name": "layer_decode", "kind": "layer", "use": "decode", "dtype": "bf16", "batch": 32, "tokens": 1,
         "heads": 16, "key_dim": 128, "value_dim": 128, "padded": False},
        # one short prompt of odd length: latency of the prefill
        {"name": "prefill_short", "kind": "prefill", "dtype": "bf16", "lengths": "333", "packed": False, "heads": 32,
         "key_dim": 128, "value_dim": 128, "state": False},
        # the long-context prefill of one sequence, continuing from a state
        {"name": "prefill_long", "kind": "prefill", "dtype": "bf16", "lengths": "8192", "packed": False, "heads": 16,
         "key_dim": 128, "value_dim": 128, "state": True},
        # a right-padded batch of ragged prompts at the smaller head size
        {"name": "prefill_padded", "kind": "prefill", "dtype": "bf16", "lengths": "1000,871,640,999,517,1000,64,333",
         "packed": False, "heads": 8, "key_dim": 64, "value_dim": 64, "state": False},
        # packed documents of very different lengths, many heads
        {"name": "prefill_packed", "kind": "prefill", "dtype": "bf16", "lengths": "16384,8191,5001,3192",
         "packed": True, "heads": 32, "key_dim": 128, "value_dim": 128, "state": False},
        # full-precision inputs (evaluation and debugging runs in f32)
        {"name": "prefill_f32", "kind": "prefill", "dtype": "f32", "lengths": "8192", "packed": False, "heads": 16,
         "key_dim": 128, "value_dim": 128, "state": True},
        # the operator's training step on one long sequence
        {"name": "train_long", "kind": "train", "dtype": "bf16", "lengths": "8192", "heads": 16, "key_dim": 128,
         "value_dim": 128, "state": True},
        # a layer's prefill of a padded batch, its cache handed on to decode
        {"name": "layer_prefill", "kind": "layer", "use": "prefill", "dtype": "bf16", "batch": 2, "tokens": 1500,
         "heads": 16, "key_dim": 128, "value_dim": 128, "padded": True},
        # a layer's training step: d_model 2048, one long sequence
        {"name": "layer_train", "kind": "layer", "use": "train", "dtype": "bf16", "batch": 1, "tokens": 8192,
         "heads": 16, "key_dim": 128, "value_dim": 128, "padded": False},
        # beam search's reorder of eight layers' caches
        {"name": "cache_reorder", "kind": "cache", "layers": 8, "batch": 64, "heads": 32, "key_dim": 128,
         "value_dim": 128},
    ]


def _spread(rng, low, high):
    """A whole number spread over the logarithm of low..high."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _head_shape(rng):
    return rng.choice([(128, 128), (128, 128), (64, 64), (64, 64), (64, 128), (96, 96), (32, 64)])


def draw(rng):
    kind = rng.choice(["decode", "prefill", "prefill", "packed", "train", "train", "layer", "layer", "cache"])
    key_dim, value_dim = _head_shape(rng)
    heads = rng.choice([4, 8, 16, 32])
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
    if kind == "decode":
        tokens = rng.choice([1, 1, 1, rng.randint(2, 8)])
        return {"kind": "decode", "dtype": dtype, "batch": _spread(rng, 1, 256), "tokens": tokens, "heads": heads,
                "key_dim": key_dim, "value_dim": value_dim, "in_place": tokens == 1 and rng.random() < 0.5}
    if kind == "cache":
        return {"kind": "cache", "layers": rng.randint(1, 8), "batch": _spread(rng, 3, 64), "heads": heads,
                "key_dim": key_dim, "value_dim": value_dim}
    if kind == "layer":
        use = rng.choice(["decode", "prefill", "train"])
        batch = _spread(rng, 4, 256) if use == "decode" else rng.randint(1, 4)
        tokens = 1 if use == "decode" else _spread(rng, 65, 8192) // batch + 1
        return {"kind": "layer", "use": use, "dtype": "bf16", "batch": batch, "tokens": tokens,
                "heads": rng.choice([4, 6, 8, 10, 12, 14, 16]), "key_dim": rng.choice([64, 128]), "value_dim": 128,
                "padded": use != "decode" and batch > 1 and rng.random() < 0.5}
    if kind == "train":
        count = rng.choice([1, 1, 2, 4])
        total = _spread(rng, 200, 131072 // heads if dtype != "f32" else 65536 // heads)
        longest = max(total // count, 33)
        lengths = [longest] * count
        if count > 1 and rng.random() < 0.5:  # right-padded
            lengths = [longest] + [rng.randint(longest // 2, longest) for _ in range(count - 1)]
        return {"kind": "train", "dtype": dtype, "lengths": ",".join(map(str, lengths)), "heads": heads,
                "key_dim": key_dim, "value_dim": value_dim, "state": rng.random() < 0.5}
    count = rng.randint(2, 12) if kind == "packed" else rng.choice([1, 1, 2, 5, 8])
    cap = 131072 if dtype == "f32" else 262144
    total = _spread(rng, 100 * count, max(cap // heads, 200 * count))
    if kind == "packed":
        shares = [rng.random() + 0.05 for _ in range(count)]
        lengths = [max(1, int(total * s / sum(shares))) for s in shares]
    else:
        longest = max(total // count, 17)
        lengths = [longest] + [rng.randint(max(1, longest // 3), longest) for _ in range(count - 1)]
    return {"kind": "prefill", "dtype": dtype, "lengths": ",".join(map(str, lengths)), "packed": kind == "packed",
            "heads": heads, "key_dim": key_dim, "value_dim": value_dim, "state": rng.random() < 0.5}


# ---- inputs -------------------------------------------------------------------


def _lengths(case):
    return [int(x) for x in case["lengths"].split(",")]


def _core(gen, batch, tokens, heads, key_dim, value_dim, dtype):
    dev = gen.device
    rnd = lambda *shape: torch.randn(*shape, generator=gen, device=dev)  # noqa: E731
    q = F.normalize(rnd(batch, tokens, heads, key_dim), dim=-1).to(dtype)
    k = F.normalize(rnd(batch, tokens, heads, key_dim), dim=-1).to(dtype)
    v = rnd(batch, tokens, heads, value_dim).to(dtype)
    channel = -7.0 * torch.rand(heads, key_dim, generator=gen, device=dev)
    g = (-5.0 * torch.sigmoid(rnd(batch, tokens, heads, key_dim) + channel)).to(dtype)
    beta = torch.sigmoid(rnd(batch, tokens, heads)).to(dtype)
    return q, k, v, g, beta


def _mask(lengths, device):
    longest = max(lengths)
    if min(lengths) == longest:
        return None
    return torch.arange(longest, device=device)[None] < torch.tensor(lengths, device=device)[:, None]


def _layer_weights(case, gen):
    """Random weights of one layer in the reference's layouts; decay biases by
    its initialisation (log-uniform dt in 1e-3..1e-1, inverse softplus)."""
    dev, dtype = gen.device, DTYPES[case["dtype"]]
    H, K, V = case["heads"], case["key_dim"], case["value_dim"]
    dm, kw, vw, rank = H * V, H * K, H * V, 128
    rnd = lambda *shape, s: (torch.randn(*shape, generator=gen, device=dev) * s).to(dtype)  # noqa: E731
    dt = torch.exp(torch.rand(H, K, generator=gen, device=dev) * math.log(100.0) + math.log(0.001))
    return {
        "q_proj": rnd(kw, dm, s=0.02), "k_proj": rnd(kw, dm, s=0.02), "v_proj": rnd(vw, dm, s=0.02),
        "q_conv": rnd(kw, CONV, s=0.3), "k_conv": rnd(kw, CONV, s=0.3), "v_conv": rnd(vw, CONV, s=0.3),
        "beta_proj": rnd(H, dm, s=0.02), "alpha_down": rnd(rank, dm, s=0.02), "alpha_up": rnd(kw, rank, s=0.1),
        "b_alpha": (dt + torch.log(-torch.expm1(-dt))).to(dtype),
        "a_log": 0.1 * torch.randn(H, generator=gen, device=dev),
        "norm_weight": (1 + 0.1 * torch.randn(H, V, generator=gen, device=dev)).to(dtype),
        "gate_proj": rnd(dm, dm, s=0.02), "output_proj": rnd(dm, dm, s=0.02),
    }


def _cache(gen, batch, heads, key_dim, value_dim, dtype):
    dev = gen.device
    rnd = lambda *shape: torch.randn(*shape, generator=gen, device=dev)  # noqa: E731
    hist = lambda width: ShortConvState(rnd(batch, CONV - 1, width).to(dtype))  # noqa: E731
    return KDAState(rnd(batch, heads, key_dim, value_dim) * STATE_STD, hist(heads * key_dim), hist(heads * key_dim),
                    hist(heads * value_dim), torch.randint(1, 4096, (batch,), generator=gen, device=dev))


def prepare(case, seed):
    dev = torch.device("cuda", torch.cuda.current_device())
    gen = torch.Generator(device=dev).manual_seed(seed)
    H, K, V = case["heads"], case["key_dim"], case["value_dim"]
    s = {"case": case}
    if case["kind"] == "cache":
        s["caches"] = [_cache(gen, case["batch"], H, K, V, torch.bfloat16) for _ in range(case["layers"])]
        s["index"] = torch.randint(0, case["batch"], (case["batch"],), generator=gen, device=dev)
        return s
    dtype = DTYPES[case["dtype"]]
    if case["kind"] == "layer":
        B, T = case["batch"], case["tokens"]
        w = _layer_weights(case, gen)
        s["x"] = torch.randn(B, T, H * V, generator=gen, device=dev).to(dtype)
        s["mask"] = _mask([T] + [T - (i + 1) * T // (2 * B) for i in range(B - 1)], dev) if case["padded"] else None
        if case["use"] == "train":
            for t in (*w.values(), s["x"]):
                t.requires_grad_()
            s["d_out"] = torch.randn(B, T, H * V, generator=gen, device=dev).to(dtype)
        s["params"] = w
        s["weights"] = KDALayerWeights(num_heads=H, key_head_dim=K, value_head_dim=V, **w)
        s["cache"] = _cache(gen, B, H, K, V, dtype) if case["use"] == "decode" else None
        return s
    if case["kind"] == "decode":
        B, T = case["batch"], case["tokens"]
        states, s["mask"], s["cu"] = B, None, None
    else:
        lengths = _lengths(case)
        packed = case.get("packed", False)
        B, T = (1, sum(lengths)) if packed else (len(lengths), max(lengths))
        states = len(lengths)
        s["mask"] = None if packed else _mask(lengths, dev)
        s["cu"] = torch.tensor([0, *lengths]).cumsum(0).to(torch.int32) if packed else None
    s["core"] = _core(gen, B, T, H, K, V, dtype)
    with_state = case["kind"] == "decode" or case["state"]
    s["state"] = torch.randn(states, H, K, V, generator=gen, device=dev) * STATE_STD if with_state else None
    if case["kind"] == "train":
        s["leaves"] = [t.requires_grad_() for t in (*s["core"], s["state"]) if t is not None]
        s["d_out"] = torch.randn(B, T, H, V, generator=gen, device=dev).to(dtype)
        if s["mask"] is not None:
            s["d_out"] *= s["mask"][:, :, None, None]
        s["d_state"] = torch.randn(states, H, K, V, generator=gen, device=dev) * STATE_STD if with_state else None
    return s


# ---- one pass -----------------------------------------------------------------

_STATE_FIELDS = ("recurrent", "q_conv", "k_conv", "v_conv", "offset")


def _state_outputs(state):
    return dict(zip(_STATE_FIELDS, (state.recurrent_state, state.q_conv_state.buffer, state.k_conv_state.buffer,
                                    state.v_conv_state.buffer, state.sequence_offset)))


def run(state):
    s, case = state, state["case"]
    if case["kind"] == "cache":
        return [_state_outputs(c) for c in reorder_states(s["caches"], s["index"])]
    if case["kind"] == "decode":
        with torch.no_grad():
            out = kda.recurrent_kda(*s["core"], s["state"], True, update_state_in_place=case["in_place"])
        return {"hidden": out.hidden_states, "state": out.final_state}
    if case["kind"] == "prefill":
        with torch.no_grad():
            out = kda.chunkwise_kda(*s["core"], s["state"], True, s["mask"], cu_seqlens=s["cu"])
        return {"hidden": out.hidden_states, "state": out.final_state}
    if case["kind"] == "train":
        with_state = s["state"] is not None
        out = kda.chunkwise_kda(*s["core"], s["state"], with_state, s["mask"])
        ends = [out.hidden_states] + ([out.final_state] if with_state else [])
        grads = torch.autograd.grad(ends, s["leaves"], [s["d_out"]] + ([s["d_state"]] if with_state else []))
        return {"hidden": ends[0].detach(), "state": ends[1].detach() if with_state else None,
                "grads": dict(zip(("q", "k", "v", "g", "beta", "state"), grads))}
    if case["use"] == "train":
        out = kda_attention_forward(s["weights"], s["x"], s["mask"], mode="chunkwise")
        names = ("x", *s["params"])
        grads = torch.autograd.grad(out.hidden_states, (s["x"], *s["params"].values()), s["d_out"])
        return {"hidden": out.hidden_states.detach(), "grads": dict(zip(names, grads))}
    with torch.no_grad():
        out = kda_attention_forward(s["weights"], s["x"], s["mask"], s["cache"],
                                    mode="decode" if case["use"] == "decode" else "chunkwise", output_final_state=True)
    return {"hidden": out.hidden_states, **_state_outputs(out.state)}


# ---- what a pass cannot do without ---------------------------------------------


def _chunk_flops(tokens_heads, K, V, C=64):
    """Causal-counted products of the chunkwise form, per token and head."""
    return tokens_heads * (6 * K * V + (3 * C + 1) * K + 2 * (C + 1) * V)


def work(case):
    H, K, V = case["heads"], case["key_dim"], case["value_dim"]
    if case["kind"] == "cache":
        rows = case["batch"] * (4 * H * K * V + 2 * (CONV - 1) * (2 * H * K + H * V) + 8)
        return {"bytes": 2 * case["layers"] * rows + 8 * case["batch"], "flops": 0}
    size = DTYPES[case["dtype"]].itemsize
    if case["kind"] == "layer":
        n, dm, kw, vw, rank = case["batch"] * case["tokens"], H * V, H * K, H * V, 128
        weights = dm * (2 * kw + vw + H + rank + 2 * dm) + kw * rank
        flops = 2 * n * weights + _chunk_flops(n * H, K, V)
        moved = size * (weights + 2 * n * dm)
        states = 4 * case["batch"] * H * K * V
        if case["use"] == "decode":
            return {"bytes": moved + 2 * states, "flops": 2 * n * weights + 8 * n * H * K * V}
        if case["use"] == "prefill":
            return {"bytes": moved + states, "flops": flops}
        # backward: x, weights and d_out read, their gradients written
        return {"bytes": 2 * moved + size * (weights + 2 * n * dm), "flops": 3 * flops}
    if case["kind"] == "decode":
        n, states, tokens_heads = case["batch"], case["batch"], case["batch"] * case["tokens"] * H
        io = size * tokens_heads * (3 * K + 2 * V + 1)
        return {"bytes": io + 8 * states * H * K * V, "flops": 8 * tokens_heads * K * V}
    lengths = _lengths(case)
    tokens_heads = sum(lengths) * H
    states = 4 * len(lengths) * H * K * V
    io = size * tokens_heads * (3 * K + 2 * V + 1)
    flops = _chunk_flops(tokens_heads, K, V)
    if case["kind"] == "prefill":
        return {"bytes": io + states * (2 if case["state"] else 1), "flops": flops}
    # forward, then inputs and d_out read and five gradients written
    back = size * tokens_heads * (6 * K + 3 * V + 2)
    return {"bytes": io + back + (5 * states if case["state"] else 0), "flops": 3 * flops}


def tolerance(case):
    """About four times the distance measured between the path and 64 bits over
    the listed and 24 drawn cases (relative 2-norm; largest difference): decode
    bf16 1.7e-3, f16 2.1e-4, f32 1e-7; operator and its gradients bf16/f16
    5e-3 (largest 5e-2), f32 8e-6 (8e-5); layer decode 3.8e-3 (3e-2), prefill
    6.2e-3 (8e-2), training 1.6e-2 (0.29)."""
    if case["kind"] == "cache":
        return "exact"
    if case["kind"] == "decode":
        return {"bf16": {"rel": 7e-3, "max": 1.6e-2}, "f16": {"rel": 1e-3, "max": 2e-3},
                "f32": {"rel": 1e-6, "max": 1e-5}}[case["dtype"]]
    if case["kind"] == "layer":
        return {"decode": {"rel": 1.6e-2, "max": 0.13}, "prefill": {"rel": 2.5e-2, "max": 0.32},
                "train": {"rel": 3e-2, "max": 0.9}}[case["use"]]
    return {"rel": 3e-5, "max": 3e-4} if case["dtype"] == "f32" else {"rel": 2e-2, "max": 0.2}


# ---- the same in 64 bits --------------------------------------------------------


class _Recurrence(torch.autograd.Function):
    """The delta rule's recurrence over [B,T,H,*] in 64 bits, token by token,
    with its adjoint from the stored states."""

    @staticmethod
    def forward(ctx, q, k, v, a, beta, s0, keep):
        B, T, H, K = q.shape
        S = s0.clone()
        out = torch.empty(B, T, H, v.shape[-1], dtype=q.dtype, device=q.device)
        states = torch.empty(T, B, H, K, v.shape[-1], dtype=q.dtype, device=q.device) if keep else None
        for t in range(T):
            if keep:
                states[t] = S
            kt = k[:, t, :, :, None]
            S = S * a[:, t, :, :, None]
            e = (v[:, t] - (S * kt).sum(2)) * beta[:, t, :, None]
            S = S + kt * e[:, :, None]
            out[:, t] = (S * q[:, t, :, :, None]).sum(2)
        ctx.save_for_backward(q, k, v, a, beta, states)
        return out, S

    @staticmethod
    def backward(ctx, d_out, dS):
        q, k, v, a, beta, states = ctx.saved_tensors
        dq, dk, dv, da, db = (torch.empty_like(t) for t in (q, k, v, a, beta))
        dS = dS.clone()
        for t in range(q.shape[1] - 1, -1, -1):
            kt, qt, at = k[:, t, :, :, None], q[:, t, :, :, None], a[:, t, :, :, None]
            S0 = states[t]
            S1 = S0 * at
            r = v[:, t] - (S1 * kt).sum(2)
            e = r * beta[:, t, :, None]
            do = d_out[:, t, :, None]
            dq[:, t] = ((S1 + kt * e[:, :, None]) * do).sum(3)
            dS = dS + qt * do
            de = (dS * kt).sum(2)
            dr = de * beta[:, t, :, None]
            db[:, t], dv[:, t] = (de * r).sum(2), dr
            dk[:, t] = (dS * e[:, :, None]).sum(3) - (S1 * dr[:, :, None]).sum(3)
            dS = dS - kt * dr[:, :, None]
            da[:, t] = (dS * S0).sum(3)
            dS = dS * at
        return dq, dk, dv, da, db, dS, None


def _recurrence(q, k, v, g, beta, s0, mask):
    """Output and final state; padded positions neither read, write nor decay."""
    if mask is not None:
        q, g = (torch.where(mask[:, :, None, None], t, 0.0) for t in (q, g))
        beta = torch.where(mask[:, :, None], beta, 0.0)
    if s0 is None:
        s0 = torch.zeros(q.shape[0], *q.shape[2:], v.shape[-1], dtype=q.dtype, device=q.device)
    keep = torch.is_grad_enabled() and any(t.requires_grad for t in (q, k, v, g, beta, s0))
    return _Recurrence.apply(q, k, v, g.exp(), beta, s0, keep)


def _conv64(x, weight, hist, heads, normalize):
    B, T, C = x.shape
    full = torch.cat((hist if hist is not None else x.new_zeros(B, CONV - 1, C), x), 1)
    y = F.silu(sum(full[:, CONV - 1 - j:CONV - 1 - j + T] * weight[:, j] for j in range(CONV)))
    y = y.reshape(B, T, heads, C // heads)
    return y / y.norm(dim=-1, keepdim=True).clamp_min(1e-6) if normalize else y


def _layer64(case, s):
    eps = torch.finfo(DTYPES[case["dtype"]]).eps
    train = case["use"] == "train"
    up = lambda t: t.detach().double().requires_grad_(train)  # noqa: E731
    w, x = {n: up(t) for n, t in s["params"].items()}, up(s["x"])
    H, K, (B, T, _) = case["heads"], case["key_dim"], x.shape
    c = s["cache"]
    hist = [None] * 3 if c is None else [b.buffer.double() for b in (c.q_conv_state, c.k_conv_state, c.v_conv_state)]
    q, k, v = (_conv64(x @ w[f"{n}_proj"].T, w[f"{n}_conv"], h, H, n != "v") for n, h in zip("qkv", hist))
    beta = torch.sigmoid(x @ w["beta_proj"].T).clamp(eps, 1 - eps)
    z = (x @ w["alpha_down"].T @ w["alpha_up"].T).reshape(B, T, H, K) + w["b_alpha"]
    g = -5.0 * torch.sigmoid(w["a_log"].exp()[:, None] * z).clamp(eps, 1 - eps)
    o, S = _recurrence(q, k, v, g, beta, None if c is None else c.recurrent_state.double(), s["mask"])
    o = o * torch.rsqrt(o.square().mean(-1, keepdim=True) + 1e-6) * w["norm_weight"]
    out = (o.reshape(B, T, -1) * torch.sigmoid(x @ w["gate_proj"].T)) @ w["output_proj"].T
    if s["mask"] is not None:
        out = out * s["mask"][..., None]
    if train:
        grads = torch.autograd.grad(out, (x, *w.values()), s["d_out"].double())
        return {"hidden": out.detach(), "grads": dict(zip(("x", *w), grads))}
    # the ShortConv histories are copies of rounded projections: no 64-bit value of their own
    return {"hidden": out, "recurrent": S, "q_conv": None, "k_conv": None, "v_conv": None, "offset": None}


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "cache":
        return None  # copies: nothing is computed
    if case["kind"] == "layer":
        with torch.set_grad_enabled(case["use"] == "train"):
            return _layer64(case, s)
    if case["kind"] == "train":
        x = [t.detach().double().requires_grad_() for t in s["leaves"]]
        out, S = _recurrence(*x[:5], x[5] if len(x) > 5 else None, s["mask"])
        ends = [out] + ([S] if len(x) > 5 else [])
        grads = torch.autograd.grad(ends, x, [s["d_out"].double()] + ([s["d_state"].double()] if len(x) > 5 else []))
        return {"hidden": out.detach(), "state": S.detach() if len(x) > 5 else None,
                "grads": dict(zip(("q", "k", "v", "g", "beta", "state"), grads))}
    with torch.no_grad():
        core = [t.double() for t in s["core"]]
        s0, mask = None if s["state"] is None else s["state"].double(), s["mask"]
        if s["cu"] is None:
            out, S = _recurrence(*core, s0, mask)
            return {"hidden": out, "state": S}
        # packed documents as one padded batch
        lengths, cu = _lengths(case), s["cu"].tolist()
        pad = lambda t: torch.nn.utils.rnn.pad_sequence([t[0, a:b] for a, b in zip(cu, cu[1:])], True)  # noqa: E731
        out, S = _recurrence(*(pad(t) for t in core), s0, _mask(lengths, core[0].device))
        return {"hidden": torch.cat([o[:n] for o, n in zip(out, lengths)])[None], "state": S}
