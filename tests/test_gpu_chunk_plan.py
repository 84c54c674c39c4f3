"""The prefill's own schedule at the sizes where it changes: sequences too few
or too short to fill the GPU are cut into segments of one or a few chunks
(``make_plan``).  Parity against the f32 oracle at the suite's 2e-2 for bf16
inputs, and against the one-segment schedule within 1e-2: each is off by one
rounding of its bf16 operands (about 5e-3 of the largest value), and the two
errors add at most."""

from __future__ import annotations

import ctypes

import pytest
import torch

import kda
from kda import _lib
from oracle import kda_oracle as ora
from tests._inputs import rel_err, workload

DEV = "cuda"


def _plan(n, total, longest, heads, K, V):
    cps, segs = ctypes.c_int64(0), ctypes.c_int64(0)
    _lib.check(_lib.load().kda_chunk_fwd_plan(n, total, longest, heads, K, V, _lib.dtype_code(torch.bfloat16),
                                              ctypes.byref(cps), ctypes.byref(segs)))
    return cps.value


def test_plan_cuts_short_and_few_sequences():
    assert _plan(1, 192, 0, 4, 128, 128) == 0  # three chunks: a cut gains under a tenth
    assert _plan(1, 333, 0, 32, 128, 128) == 1
    assert _plan(1, 4096, 0, 4, 128, 128) == 2
    assert _plan(4, 4 * 64, 0, 64, 128, 128) == 0  # single chunks
    assert _plan(8, 8 * 2048, 0, 32, 128, 128) == 0  # one chain per CU
    # the schedules whose workspace the fixed-scratch entry point must hold
    for heads in (1, 8, 64, 191):
        for tokens in range(64, 4096, 192):
            need = _lib.load().kda_chunk_fwd_workspace_bytes(1, tokens, 0, heads, 128, 256, 2)
            assert tokens // 64 * heads * 2 >= 512 or need <= _lib.NOALLOC_SCRATCH_BYTES


def test_plan_of_uneven_documents_fills_whole_rounds():
    """Known longest document: the segments of two documents, whose lengths the
    hint gives exactly, fit whole rounds of 256 workgroups; degenerate sizes
    plan without a cut."""
    for heads, long, short in ((4, 9000, 3000), (8, 20000, 5000), (16, 6393, 3416), (32, 6000, 1000)):
        cut = _plan(2, long + short, long, heads, 64, 64)
        n, m = -(-long // 64), -(-short // 64)
        workgroups = (-(-n // cut) - (-m // cut)) * heads
        assert cut >= 1 and 1 <= -(-workgroups // 256) <= 4
        shorter = (-(-n // (cut - 1)) - (-m // (cut - 1))) * heads
        assert -(-shorter // 256) > -(-workgroups // 256), (heads, cut)  # the shortest that fits
    assert _plan(256, 300, 45, 32, 128, 128) == 0  # more documents than rounds have room for
    assert _plan(2, 1, 1, 4, 128, 128) == 0  # an empty document


@pytest.mark.gpu
@pytest.mark.parametrize(
    "B,T,H,K,V,docs",
    [
        (1, 256, 2, 128, 128, None),   # four whole chunks, one a segment
        (1, 257, 2, 64, 64, None),     # a last chunk of one token
        (1, 1100, 8, 128, 128, None),  # several chunks a segment, a partial last one
        (3, 600, 24, 128, 128, None),  # as many segments as the CUs take in one round
        (1, 450, 3, 96, 256, None),    # two column groups, padded key channels
        (1, 901, 4, 128, 128, [0, 1, 65, 129, 900, 901]),  # packed: single tokens beside a long document
        (1, 5000, 4, 64, 64, [0, 1130, 1131, 3000, 4999, 5000]),  # single tokens, several chunks a segment
        (1, 3300, 16, 128, 128, [0, 2111, 2500, 3300]),  # segments of several chunks, 16 heads
    ],
)
def test_planned_schedule_matches_oracle(segments, B, T, H, K, V, docs):
    q, k, v, g, beta, _ = workload(B, T, H, K, V, seed=31)
    n = B if docs is None else len(docs) - 1
    longest = 0 if docs is None else max(b - a for a, b in zip(docs, docs[1:]))
    assert _plan(n, B * T, longest, H, K, V) >= 1
    state = torch.randn(n, H, K, V, generator=torch.Generator().manual_seed(32)) * 0.02
    ins = [t.to(DEV) for t in (q, k, v, g, beta, state)]
    got = kda.chunkwise_kda(*ins, True, cu_seqlens=docs)
    segments(0)
    one = kda.chunkwise_kda(*ins, True, cu_seqlens=docs)
    f = [t.float() for t in (q, k, v, g, beta)]
    if docs is None:
        ro, rs = ora.chunkwise(*f, state, chunk_size=64, secondary_tile_size=16)
    else:
        ro, rs = ora.varlen_chunkwise(*f, docs, state)
    assert rel_err(got.hidden_states, ro) < 2e-2 and rel_err(got.final_state, rs) < 2e-2
    assert rel_err(got.hidden_states, one.hidden_states) < 1e-2
    assert rel_err(got.final_state, one.final_state) < 1e-2
