"""Which decode steps of a layer take the three-launch path by size: calls of
large layers and batches, whose projections read their weights once for every
64 sequences, keep the composed stages."""

from __future__ import annotations

import pytest
import torch

from kda import layer
from kda.layer import KDALayerWeights


def _weights(d_model, rank=128):
    H = d_model // 128
    t = lambda *s: torch.empty(*s, dtype=torch.bfloat16, device="meta")  # noqa: E731
    sq = lambda: t(d_model, d_model)  # noqa: E731
    return KDALayerWeights(num_heads=H, key_head_dim=128, value_head_dim=128, q_proj=sq(), k_proj=sq(), v_proj=sq(),
                           q_conv=t(d_model, 4), k_conv=t(d_model, 4), v_conv=t(d_model, 4), beta_proj=t(H, d_model),
                           alpha_down=t(rank, d_model), alpha_up=t(d_model, rank), b_alpha=t(H, 128), a_log=t(H),
                           norm_weight=None, gate_proj=sq(), output_proj=sq())


@pytest.mark.parametrize("d_model,batch,native", [(512, 256, True), (2048, 1, True), (2048, 256, True), (4096, 65, True),
                                                  (4096, 128, False), (4096, 256, False), (7168, 4, True),
                                                  (7168, 64, False)])
def test_size_rule_follows_the_measured_sides(d_model, batch, native):
    assert layer._few_products(_weights(d_model), batch) is native


@pytest.mark.parametrize("d_model,batch,composed", [(1024, 256, False), (1536, 192, True), (2048, 128, False),
                                                    (2048, 129, True), (2048, 256, True), (3072, 64, False),
                                                    (3072, 96, True), (4096, 48, False), (4096, 64, True),
                                                    (6144, 24, False), (7168, 16, False), (7168, 24, True)])
def test_captured_calls_follow_the_device_times(monkeypatch, d_model, batch, composed):
    w = _weights(d_model)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert layer._captured_past_the_line(w, batch) is composed
    w.key_head_dim = 64  # the composed stages are slower at every such size
    assert layer._captured_past_the_line(w, batch) is False
    w.key_head_dim = 128
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert layer._captured_past_the_line(w, batch) is False
