"""Right-padding masks on the GPU (kda_mask_lengths): lengths, the reference's
errors in its order, and the calls that take them, against the same mask in host
memory (checked with tensor operations)."""

from __future__ import annotations

import pytest
import torch

import kda
from kda import fused
from kda.layer import KDALayerWeights, kda_attention_forward
from kda.utils import checked_lengths, validate_attention_mask
from tests._inputs import layer_weights, workload

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda")


def _mask(lengths, tokens):
    return torch.arange(tokens)[None] < torch.tensor(lengths)[:, None]


@pytest.mark.parametrize("tokens", [1, 2, 63, 64, 65, 255, 256, 257, 1000])
def test_lengths_at_wave_and_block_edges(tokens):
    lengths = sorted({1, max(1, tokens // 2), max(1, tokens - 1), tokens})
    mask = _mask(lengths, tokens).to(DEV)
    got = checked_lengths(mask, len(lengths), tokens, DEV)
    assert got.dtype == torch.int32 and got.tolist() == lengths
    wide = torch.zeros(len(lengths), 2 * tokens, dtype=torch.bool, device=DEV)
    wide[:, ::2] = mask  # a strided view
    assert checked_lengths(wide[:, ::2], len(lengths), tokens, DEV).tolist() == lengths
    assert validate_attention_mask(mask, len(lengths), tokens) is mask


def test_errors_like_a_host_mask():
    ok = _mask([3, 5], 5)
    hole, empty = ok.clone(), ok.clone()
    hole[0, 1] = False
    empty[1] = False
    both = hole.clone()
    both[1] = False
    late = torch.zeros(1, 300, dtype=torch.bool)
    late[0, 299] = True  # valid tokens in another wave than the padding before them
    for mask, text in ((hole, "monotonic"), (empty, "all-padding"), (both, "monotonic"), (late, "monotonic")):
        for m in (mask, mask.to(DEV)):
            with pytest.raises(ValueError, match=text):
                validate_attention_mask(m, *m.shape)
            with pytest.raises(ValueError, match=text):
                checked_lengths(m, *m.shape, DEV)
    with pytest.raises(ValueError, match="shape"):
        checked_lengths(ok.to(DEV), 2, 6, DEV)
    with pytest.raises(TypeError, match="boolean"):
        checked_lengths(ok.to(DEV).int(), 2, 5, DEV)
    assert validate_attention_mask(empty.to(DEV), 2, 5, require_nonempty=False) is not None


def test_operators_take_device_and_host_masks_alike():
    q, k, v, g, beta, _ = (None if t is None else t.to(DEV) for t in workload(2, 130, 2, 64, 64, seed=4))
    mask = _mask([130, 71], 130)
    for fn in (kda.chunkwise_kda, kda.recurrent_kda):
        a, b = (fn(q, k, v, g, beta, None, True, m) for m in (mask, mask.to(DEV)))
        assert torch.equal(a.hidden_states, b.hidden_states) and torch.equal(a.final_state, b.final_state)
    x = torch.randn(2, 130, 128, generator=torch.Generator().manual_seed(1)).to(DEV, torch.bfloat16)
    w = torch.randn(128, 4, generator=torch.Generator().manual_seed(2)).to(DEV, torch.bfloat16)
    a, b = (fused.conv_silu(x, w, None, None, m, num_heads=2, normalize=True, output_final_state=True)
            for m in (mask, mask.to(DEV)))
    assert torch.equal(a[0], b[0]) and torch.equal(a[1].buffer, b[1].buffer)


@pytest.mark.parametrize("mode", ["chunkwise", "recurrent"])
def test_layer_with_state_and_mask_offsets(mode):
    w = layer_weights(128, 2, 64, 64, rank=16, dtype=torch.bfloat16)
    gw = KDALayerWeights(**{n: (t.to(DEV) if isinstance(t, torch.Tensor) else t) for n, t in w.items()})
    x = torch.randn(3, 70, 128, generator=torch.Generator().manual_seed(7)).to(DEV, torch.bfloat16)
    mask = _mask([70, 1, 33], 70).to(DEV)
    with torch.no_grad():
        one = kda_attention_forward(gw, x, mask, mode=mode, output_final_state=True)
        two = kda_attention_forward(gw, x, mask, one.state, mode=mode, output_final_state=True)
        bare = kda_attention_forward(gw, x, None, one.state, mode=mode, output_final_state=True)
    assert one.state.sequence_offset.tolist() == [70, 1, 33]
    assert two.state.sequence_offset.tolist() == [140, 2, 66] and two.state.sequence_offset.dtype == torch.long
    assert bare.state.sequence_offset.tolist() == [140, 71, 103]
    assert not one.hidden_states[~mask].any()
    # a row alone, without padding, gives the same rows (the same kernels on the same values)
    with torch.no_grad():
        solo = kda_attention_forward(gw, x[2:3, :33], mode=mode, output_final_state=True)
    diff = (one.hidden_states[2, :33].float() - solo.hidden_states[0].float()).abs().max()
    assert diff <= 2e-2 * solo.hidden_states.float().abs().max()
