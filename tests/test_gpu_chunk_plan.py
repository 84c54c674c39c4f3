"""The prefill's own schedule at the sizes where it changes: sequences too few
or too short to fill the GPU are cut into segments of one or a few chunks
(``make_plan``).  Parity against the f32 oracle at the suite's 2e-2 for bf16
inputs, and against the one-segment schedule within 1e-2: each is off by one
rounding of its bf16 operands (about 5e-3 of the largest value), and the two
errors add at most."""

from __future__ import annotations

import ctypes
import random

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


def _balanced_bytes(n, total, longest, heads, V):
    """Workspace of one balanced pass over 256 CUs (segments of as many chunks
    as there are chunk steps per CU; one segment per sequence where that fills
    the GPU): what the fixed-scratch entry point has to be able to plan with."""
    groups, chunks = -(-V // 128), total // 64 + n
    work = total // 64 * heads * groups
    steps = -(-work // 256)
    uneven = n > 1 and 4 * -(-longest // 64) > 5 * steps
    maps = (2 * (n + 1) * 4 + 255) // 256 * 256
    if work < 512 or not (uneven or 4 * n * heads * groups < 768):
        return maps
    segs = chunks // steps + n + 1
    return maps + heads * (segs * (2 * 4 * 128 * V + 2 * 128 * 128) + chunks * 12 * 1024)


@pytest.mark.parametrize("packed", [False, True])
@pytest.mark.parametrize("V", [64, 128, 256])
def test_fixed_scratch_holds_what_one_balanced_pass_fits(packed, V):
    """kda_chunk_fwd_noalloc takes every call whose fastest schedule or whose
    balanced pass fits its scratch, and refuses the others.  (The size check
    comes before the pointers are looked at; the null pointers then end the call
    before anything is launched.)"""
    lib, bf16, rng = _lib.load(), _lib.dtype_code(torch.bfloat16), random.Random(V + packed)
    calls = [(1, 2016, 2016, 96), (3, 3 * 1998, 1998, 32), (1, 2012, 2012, 48), (24, 24 * 2036, 2036, 4),
             (13, 20528, 2711, 12), (1, 262144, 262144, 16)]
    for _ in range(3000):
        n, heads = rng.randint(1, 24), rng.choice([1, 2, 3, 4, 8, 12, 16, 24, 32, 48, 64, 96, 128, 190])
        longest = int(2 ** rng.uniform(6, 14))
        total = n * longest if not packed else longest + sum(rng.randint(1, longest) for _ in range(n - 1))
        calls.append((n, total, longest, heads))
    taken = {True: 0, False: 0}
    for n, total, longest, heads in calls:
        if not packed:
            total = n * longest
        hint = longest if packed else 0
        query = lib.kda_chunk_fwd_workspace_bytes(n, total, hint, heads, 128, V, bf16)
        fits = min(query, _balanced_bytes(n, total, hint, heads, V)) <= _lib.NOALLOC_SCRATCH_BYTES
        status = lib.kda_chunk_fwd_noalloc(None, None, None, None, None, bf16, None, None, 0, None,
                                           16 if packed else None, longest, None, n, total, heads, 128, V, None)
        assert status != _lib.KDA_OK
        assert (status != _lib.KDA_ERR_WORKSPACE) == fits, (n, total, longest, heads)
        taken[fits] += 1
    assert min(taken.values()) >= 5


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


@pytest.mark.gpu
@pytest.mark.parametrize("B,T,H,V,docs", [
    (24, 2036, 4, 128, None),  # the fastest schedule takes 175 MiB, the balanced pass 93
    (1, 2012, 48, 256, None),  # 153 against 72 MB
    (1, 20528, 12, 128, [0, 2711, *(2711 + 1485 * i for i in range(1, 12)), 20528]),  # 176 against 114 MiB
])
def test_schedule_within_a_smaller_workspace_matches(B, T, H, V, docs):
    """The balanced pass that a smaller workspace gets (the fixed scratch, or a
    caller's own) against the fastest schedule, within the module's 1e-2."""
    lib, bf16 = _lib.load(), _lib.dtype_code(torch.bfloat16)
    q, k, v, g, beta, _ = workload(B, T, H, 128, V, seed=33)
    n = B if docs is None else len(docs) - 1
    span = T if docs is None else max(b - a for a, b in zip(docs, docs[1:]))
    hint = 0 if docs is None else span
    need = lib.kda_chunk_fwd_workspace_bytes(n, B * T, hint, H, 128, V, bf16)
    small = _balanced_bytes(n, B * T, hint, H, V)
    assert small <= _lib.NOALLOC_SCRATCH_BYTES < need
    ins = [t.to(DEV) for t in (q, k, v, g, beta)]
    s0 = torch.randn(n, H, 128, V, generator=torch.Generator().manual_seed(34)).mul_(0.02).to(DEV)
    cu = None if docs is None else torch.tensor(docs, dtype=torch.int32, device=DEV)
    stream = torch.cuda.current_stream().cuda_stream
    got = []
    for room in (need, small, None):
        out = torch.full((B, T, H, V), float("nan"), dtype=torch.bfloat16, device=DEV)
        final = torch.full((n, H, 128, V), float("nan"), device=DEV)
        args = (*(t.data_ptr() for t in ins), bf16, s0.data_ptr(), final.data_ptr(), 0, out.data_ptr(), _lib.ptr(cu),
                span, None, n, B * T, H, 128, V)
        if room is None:
            _lib.check(lib.kda_chunk_fwd_noalloc(*args, stream))
        else:
            ws = torch.empty(room, dtype=torch.uint8, device=DEV)
            _lib.check(lib.kda_chunk_fwd(*args, ws.data_ptr(), room, stream))
            assert lib.kda_chunk_fwd(*args, ws.data_ptr(), small - 1, stream) == _lib.KDA_ERR_WORKSPACE
        got.append((out, final))
    for out, final in got[1:]:
        assert rel_err(out, got[0][0]) < 1e-2 and rel_err(final, got[0][1]) < 1e-2
    assert torch.equal(got[1][0], got[2][0]) and torch.equal(got[1][1], got[2][1])  # one schedule, the same bits
