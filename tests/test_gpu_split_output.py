"""The split-bf16 chunk path's output reruns at the edges of chunks, segments
and value tiles: f32 inputs against the f64 scalar recurrence.  An output passes
through at most three split records in one term (K~, W and Qg, or Aqk), each
within 2^-17 of its value: 3 x 7.6e-6 of the largest output."""

from __future__ import annotations

import pytest
import torch

import kda
from oracle import c_oracle
from tests._inputs import rel_err, workload

pytestmark = pytest.mark.gpu
TOL = 3 * 2.0**-17


@pytest.mark.parametrize(
    "B,T,H,K,V",
    [
        (1, 1, 1, 128, 128),   # one position
        (1, 63, 2, 128, 128),  # a chunk short of one row
        (1, 65, 2, 64, 64),    # a second chunk of one row
        (2, 129, 3, 128, 1),   # one value column
        (1, 200, 2, 72, 33),   # a column past two value tiles
        (1, 97, 2, 33, 31),    # odd row stride
        (1, 1000, 4, 128, 96),  # many segments, six of eight waves with columns
        (3, 321, 96, 64, 17),  # more chains than CUs: one segment each
    ],
)
def test_output_reruns_match_f64_recurrence(B, T, H, K, V):
    q, k, v, g, beta, state = workload(B, T, H, K, V, state_std=0.02, seed=71, dtype=torch.float32)
    got = kda.chunkwise_kda(*(t.to("cuda") for t in (q, k, v, g, beta, state)), True)
    ro, rs = c_oracle.recurrent_ref(q, k, v, g, beta, state)
    assert rel_err(got.hidden_states, ro) < TOL and rel_err(got.final_state, rs) < TOL
