"""The chunk backward where beta is zero: the beta gradient is E . e with e the
delta rule's error, which the pseudo-value Vt = beta e no longer carries, so
those rows take it from the records directly.  Against the f64 oracle at the
suite's tolerances (f32 2e-4, bf16 2e-2 of each gradient's largest value)."""

from __future__ import annotations

import pytest
import torch

import kda
from kda import _lib
from oracle import kda_oracle as ora
from tests._inputs import rel_err, workload

pytestmark = pytest.mark.gpu
DEV = "cuda"
TOL = {torch.float32: 2e-4, torch.bfloat16: 2e-2, torch.float16: 2e-2}


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,H,K,V", [(1, 65, 2, 128, 128), (2, 191, 2, 64, 64), (1, 130, 1, 40, 50),
                                       (1, 1024, 1, 128, 128)])
@pytest.mark.parametrize("zeros", ["first", "some", "chunk", "all"])
def test_beta_gradient_at_zero_beta(dtype, B, T, H, K, V, zeros):
    q, k, v, g, beta, s0 = workload(B, T, H, K, V, state_std=0.5, g_shift=0.0, seed=T + K, dtype=dtype)
    gen = torch.Generator().manual_seed(5)
    if zeros == "first":
        beta[:, 0] = 0
    elif zeros == "some":
        beta[torch.rand(B, T, H, generator=gen) < 0.3] = 0
        if dtype != torch.float16:
            beta[:, 1] = 1e-36  # its Vt is no f32 operand either
    elif zeros == "chunk":
        beta[:, 16:80] = 0
    else:
        beta[:] = 0
    d_out = torch.randn(B, T, H, V, generator=gen).to(dtype)
    d_final = torch.randn(B, H, K, V, generator=gen)
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v, g, beta, s0)]
    res = kda.chunkwise_kda(*leaves, True)
    got = torch.autograd.grad([res.hidden_states, res.final_state], leaves, [d_out.to(DEV), d_final.to(DEV)])
    ref = ora.chunkwise_backward(*(t.double() for t in (q, k, v, g, beta, s0)), d_out.double(), d_final.double(),
                                 chunk_size=64)
    for name, a, r in zip(("dq", "dk", "dv", "dg", "dbeta", "ds0"), got, ref):
        assert torch.isfinite(a).all(), name
        if float(r.abs().max()) > 1e-30:
            assert rel_err(a, r) < TOL[dtype], (name, rel_err(a, r))
        else:
            assert float(a.abs().max()) < 1e-30, name


@pytest.mark.parametrize("dtype,K,V", [(torch.bfloat16, 128, 128), (torch.float32, 64, 48)])
@pytest.mark.parametrize("zeros", [0, 1])
def test_positions_past_the_end_are_no_zero_beta_rows(dtype, K, V, zeros):
    """Only a chunk with a real row of zero beta forms those rows' records, for
    which alone its A (floats 4096 .. 8191 of the chunk's workspace record) is
    written: the positions past the sequence's end have no beta gradient."""
    T, H, lib, code = 65, 3, _lib.load(), _lib.dtype_code(dtype)
    q, k, v, g, beta, _ = (None if t is None else t.to(DEV) for t in workload(1, T, H, K, V, seed=8, dtype=dtype))
    beta[0, T - 1, 1] *= 1 - zeros  # the last chunk's only row, second head
    need = lib.kda_chunk_bwd_workspace_bytes(1, T, H, K, V, code)
    ws = torch.full((need // 4,), float("nan"), device=DEV)
    grads = [torch.empty_like(t) for t in (q, k, v, g, beta)]
    _lib.check(lib.kda_chunk_bwd(*(t.data_ptr() for t in (q, k, v, g, beta, torch.ones_like(v))), code, None, None,
                                 *(t.data_ptr() for t in grads), None, 1, T, H, K, V, ws.data_ptr(), need,
                                 torch.cuda.current_stream().cuda_stream))
    assert all(torch.isfinite(t).all() for t in grads)
    Kp, Vp, s = 64 if K <= 64 else 128, -(-V // 32) * 32, 1 if dtype == torch.float32 else 2
    rec = 2 * 4096 + 4096 // s + 5 * 64 * Kp // s + 2 * 64 * Vp + Kp + 64 + (2 * Kp * Vp + 64 * Vp) // s
    records = ws[: 2 * H * (-(-rec // 64) * 64)].reshape(H, 2, -1)  # (head, chunk)
    written = ~records[:, :, 4096:8192].isnan().all(dim=2)
    assert written.tolist() == [[False, False], [False, bool(zeros)], [False, False]]
