"""The native decode step of a layer (kda_layer_decode) at its edges: batches
around the 16-row tiles, d_model of one slice, every head shape, taps and rank
limits, missing state, biases and norm weights.  Against the oracle layer at the
suite's 2e-2 (bf16 and f16 activations, max|x - ref| / max|ref|), with the
histories, which are rounded projections, within 1e-2; and against the composed
stages, which round at the same points and differ by the order of f32 sums
before a rounding: one unit in the last place of the largest value (2^-8)
through two rounded products, 1e-2."""

from __future__ import annotations

import pytest
import torch

import kda
from kda import layer
from kda.layer import KDALayerWeights, kda_attention_forward
from oracle import kda_oracle as ora
from tests._inputs import layer_weights, rel_err

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _case(B, H, K, V, taps, rank, dtype, biases, norm, seed):
    w = layer_weights(H * V, H, K, V, conv=taps, rank=rank, dtype=dtype, seed=seed, biases=biases)
    if norm == "shared":
        w["norm_weight"] = w["norm_weight"][0].contiguous()
    elif norm is None:
        w["norm_weight"] = None
    gen = torch.Generator().manual_seed(seed + 1)
    x = torch.randn(B, 1, H * V, generator=gen).to(dtype)
    hist = lambda n: torch.randn(B, taps - 1, n, generator=gen).to(dtype)  # noqa: E731
    st = (torch.randn(B, H, K, V, generator=gen) * 0.1, hist(H * K), hist(H * K), hist(H * V),
          torch.arange(B, dtype=torch.long) + 5)
    gw = KDALayerWeights(**{k: (v.to(DEV) if isinstance(v, torch.Tensor) else v) for k, v in w.items()})
    return w, gw, x, st


def _state(st):
    return kda.KDAState(st[0].to(DEV), *(kda.ShortConvState(t.to(DEV)) for t in st[1:4]), st[4].to(DEV))


def _tuple(s):
    return (s.recurrent_state, s.q_conv_state.buffer, s.k_conv_state.buffer, s.v_conv_state.buffer, s.sequence_offset)


@pytest.mark.parametrize("B,H,K,V,taps,rank,dtype,biases,norm,with_state", [
    (1, 1, 64, 64, 4, 8, torch.bfloat16, False, "head", True),    # one slice of d_model, one head
    (15, 2, 128, 128, 4, 128, torch.bfloat16, False, "head", True),
    (17, 3, 64, 128, 4, 32, torch.float16, True, "shared", True),  # a second row tile, one row in it
    (33, 2, 128, 64, 2, 256, torch.bfloat16, True, None, True),
    (64, 5, 64, 64, 8, 200, torch.bfloat16, False, "head", False),
    (65, 2, 128, 128, 4, 64, torch.bfloat16, True, "head", False),  # a second block of 64 sequences
    (256, 9, 64, 64, 3, 16, torch.float16, False, "head", True),
    (3, 16, 128, 128, 4, 128, torch.bfloat16, False, "head", True),
])
def test_native_decode_step(monkeypatch, B, H, K, V, taps, rank, dtype, biases, norm, with_state):
    w, gw, x, st = _case(B, H, K, V, taps, rank, dtype, biases, norm, seed=B + K)
    step = layer._decode_step
    taken = []
    monkeypatch.setattr(layer, "_decode_step", lambda *a: taken.append(step(*a)) or taken[-1])
    with torch.no_grad():
        got = kda_attention_forward(gw, x.to(DEV), state=_state(st) if with_state else None, mode="decode")
    assert taken[0] is not None
    monkeypatch.setattr(layer, "DECODE_STEP_BATCH", 0)
    with torch.no_grad():
        ref = kda_attention_forward(gw, x.to(DEV), state=_state(st) if with_state else None, mode="decode")
    assert taken[1] is None
    ro, rst = ora.kda_layer(w, x, None, st if with_state else None, mode="decode")
    assert got.hidden_states.dtype == dtype and got.hidden_states.shape == ref.hidden_states.shape
    assert rel_err(got.hidden_states, ro) < 2e-2 and rel_err(got.hidden_states, ref.hidden_states) < 1e-2
    for i, (a, b, c) in enumerate(zip(_tuple(got.state), rst, _tuple(ref.state))):
        assert a.dtype == c.dtype and a.shape == c.shape
        if i == 4:
            assert a.tolist() == b.tolist() == c.tolist()
        elif a.numel():
            assert rel_err(a, b) < (2e-2 if i == 0 else 1e-2) and rel_err(a, c) < 1e-2, i


def test_native_decode_step_in_place_and_inputs_untouched():
    w, gw, x, st = _case(4, 2, 128, 128, 4, 32, torch.bfloat16, False, "head", seed=9)
    state, xd = _state(st), x.to(DEV)
    before = [t.clone() for t in _tuple(state)]
    with torch.no_grad():
        new = kda_attention_forward(gw, xd, state=state, mode="decode")
        assert all(torch.equal(a, b) for a, b in zip(before, _tuple(state)))
        same = kda_attention_forward(gw, xd, state=state, mode="decode", update_state_in_place=True)
    assert same.state.recurrent_state.data_ptr() == state.recurrent_state.data_ptr()
    assert torch.equal(same.state.recurrent_state, new.state.recurrent_state)
    assert torch.equal(same.hidden_states, new.hidden_states)


def test_calls_the_native_step_leaves_to_the_stages():
    # autograd, a weight in another dtype, autocast and a wrong state keep the
    # composed stages and their errors
    w, gw, x, st = _case(2, 2, 64, 64, 4, 16, torch.bfloat16, False, "head", seed=3)
    xd, state = x.to(DEV), _state(st)
    assert layer._decode_step(gw, xd, state, False) is not None
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert layer._decode_step(gw, xd, state, False) is None
    assert layer._decode_step(gw, xd.requires_grad_(), state, False) is None
    out = kda_attention_forward(gw, xd, state=state, mode="decode")
    assert out.hidden_states.requires_grad
    xd = xd.detach()
    gw.b_alpha = gw.b_alpha.float()
    assert layer._decode_step(gw, xd, state, False) is None
    gw.b_alpha = gw.b_alpha.bfloat16()
    gw.q_conv = gw.q_conv.float()
    with pytest.raises(TypeError, match="weight must have dtype"), torch.no_grad():
        kda_attention_forward(gw, xd, state=state, mode="decode")


@pytest.mark.parametrize("B,native", [(32, True), (256, False)])
def test_captured_step_takes_the_faster_route_and_replays(monkeypatch, B, native):
    # a large batch: the native step outside a capture, the composed stages
    # (faster without their host time) inside one; each replay after other work
    w, gw, x, st = _case(B, 16, 128, 128, 4, 128, torch.bfloat16, False, "head", seed=B)
    xd, state, step, taken = x.to(DEV), _state(st), layer._decode_step, []
    monkeypatch.setattr(layer, "_decode_step", lambda *a: taken.append(step(*a)) or taken[-1])
    with torch.no_grad():
        ref = kda_attention_forward(gw, xd, state=state, mode="decode")
        assert taken.pop() is not None
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            monkeypatch.setattr(layer, "DECODE_STEP_BATCH", 0 if not native else 256)  # the route to be captured
            kda_attention_forward(gw, xd, state=state, mode="decode")
        torch.cuda.current_stream().wait_stream(side)
        monkeypatch.setattr(layer, "DECODE_STEP_BATCH", 256)
        taken.clear()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            got = kda_attention_forward(gw, xd, state=state, mode="decode")
        assert (taken.pop() is not None) is native
        for seed in range(3):
            xd.copy_(torch.randn(x.shape, generator=torch.Generator().manual_seed(seed)))
            ref = kda_attention_forward(gw, xd, state=state, mode="decode")  # eager work between the replays
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert rel_err(got.hidden_states, ref.hidden_states) < 1e-2
            for i, (a, b) in enumerate(zip(_tuple(got.state), _tuple(ref.state))):
                assert torch.equal(a, b) if i == 4 or native else rel_err(a, b) < 1e-2, i


def test_a_layer_without_decay_bias_keeps_the_stages():
    w, gw, x, st = _case(3, 2, 64, 64, 4, 16, torch.bfloat16, False, "head", seed=4)
    gw.b_alpha = torch.zeros_like(gw.b_alpha)
    with torch.no_grad():
        ref = kda_attention_forward(gw, x.to(DEV), state=_state(st), mode="decode")
        gw.b_alpha = None
        got = kda_attention_forward(gw, x.to(DEV), state=_state(st), mode="decode")
    assert rel_err(got.hidden_states, ref.hidden_states) < 1e-2
    assert rel_err(got.state.recurrent_state, ref.state.recurrent_state) < 1e-2


@pytest.mark.parametrize("transform", ["vmap", "dual"])
def test_transforms_of_the_output_projection_keep_the_stages(transform):
    # the output projection is torch's linear: it takes batched and dual weights
    w, gw, x, st = _case(3, 2, 64, 64, 4, 16, torch.bfloat16, False, "head", seed=6)
    xd, state, weight = x.to(DEV), _state(st), gw.output_proj
    other = torch.randn(weight.shape, generator=torch.Generator().manual_seed(2)).to(weight)

    def call(m):
        gw.output_proj = m
        return kda_attention_forward(gw, xd, state=state, mode="decode").hidden_states

    with torch.no_grad():
        one, two = call(weight), call(other)
        if transform == "vmap":
            both = torch.vmap(call)(torch.stack([weight, other]))
            assert rel_err(both[0], one) < 1e-2 and rel_err(both[1], two) < 1e-2
        else:
            with torch.autograd.forward_ad.dual_level():
                got = torch.autograd.forward_ad.unpack_dual(
                    call(torch.autograd.forward_ad.make_dual(weight, other)))
            assert rel_err(got.primal, one) < 1e-2 and rel_err(got.tangent, two) < 1e-2
