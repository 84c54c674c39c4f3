"""The chunk backward where beta is zero: the beta gradient is E . e with e the
delta rule's error, which the pseudo-value Vt = beta e no longer carries, so
those rows take it from the records directly.  Against the f64 oracle at the
suite's tolerances (f32 2e-4, bf16 2e-2 of each gradient's largest value)."""

from __future__ import annotations

import pytest
import torch

import kda
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
