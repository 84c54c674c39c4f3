"""The split-bf16 chunk path's output reruns at the edges of chunks, segments
and value tiles: f32 inputs against the f64 scalar recurrence.  The tolerance is
empirical: the path's products, from prep's decay products to the scan's maps and
reruns, keep their operands to about 2^-17, and over these shapes and five seeds
the largest error is 1.5e-5 of the largest output and 1.9e-5 of the largest state;
2.3e-5 leaves it a quarter."""

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
