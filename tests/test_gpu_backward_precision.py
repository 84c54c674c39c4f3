"""Products of the chunk backward whose operands' rounding is visible alone:
inputs for which every other product is exact to f32, against 64 bits."""

from __future__ import annotations

import pytest
import torch

import kda
from oracle import kda_oracle as ora

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _gradients(q, k, v, g, beta, d_out):
    """Input gradients on the GPU and in 64 bits."""
    leaves = [t.to(DEV).requires_grad_() for t in (q, k, v, g, beta)]
    out = kda.chunkwise_kda(*leaves, None, False).hidden_states
    got = torch.autograd.grad(out, leaves, d_out.to(DEV))
    ref = ora.chunkwise_backward(*(t.double() for t in (q, k, v, g, beta)), None, d_out.double(), None)
    return got, ref


def _rel(a, b):
    return float((a.double().cpu() - b).norm() / b.norm())


def strict_product_error(K, V, T=64):
    """dk in the channels that only dA = -strict(dv Vt^T) reaches: q is one
    channel of the last row, g and the start state are zero, and k in that
    channel is a power of two, so that dVt is exact."""
    gen = torch.Generator().manual_seed(K + V)
    B, H, h = 2, 8, torch.float16
    k = torch.nn.functional.normalize(torch.randn(B, T, H, K, generator=gen), dim=-1).to(h)
    k[..., 0] = 0.125 * (1 - 2 * torch.randint(0, 2, (B, T, H), generator=gen))
    q = torch.zeros(B, T, H, K, dtype=h)
    q[:, -1, :, 0] = 1
    v = torch.randn(B, T, H, V, generator=gen).to(h)
    beta = torch.sigmoid(torch.randn(B, T, H, generator=gen)).to(h)
    d_out = torch.randn(B, T, H, V, generator=gen).bfloat16().to(h)
    got, ref = _gradients(q, k, v, torch.zeros_like(q), beta, d_out)
    return _rel(got[1][..., 1:], ref[1][..., 1:])


@pytest.mark.parametrize("K,V,T", [(128, 128, 64), (64, 64, 64), (96, 40, 51)])
def test_strict_product_rounds_one_operand(K, V, T):
    """f16 inputs: Vt's bf16 record is the one rounded operand.  Rounding to
    bf16 errs by 2^-8/sqrt(3) of a value's binade in the mean square, 1.5e-3 to
    1.8e-3 of the values' norm; two rounded operands err by sqrt(2) as much, from
    2.1e-3 on."""
    assert strict_product_error(K, V, T) < 2.0e-3


def beta_gradient_error(H):
    """dbeta = dO v of single tokens with q = k one channel: v and dO are bf16
    values and beta has 16 significant bits, so that Vt = beta v is exact in f32
    and no nearer than 2^-18 in two bf16 parts."""
    gen = torch.Generator().manual_seed(H)
    B, K = 8, 64
    k = torch.zeros(B, 1, H, K)
    k[..., 3] = 1
    v, d_out = (torch.randn(B, 1, H, 1, generator=gen).bfloat16().float() for _ in range(2))
    beta = torch.randint(2**15, 2**16, (B, 1, H), generator=gen).float() / 2**16
    got, ref = _gradients(k.clone(), k, v, torch.zeros_like(k), beta, d_out)
    return _rel(got[4], ref[4])


def test_f32_beta_gradient_reads_every_bit_of_vt():
    """f32 inputs: one product, one division and no operand's rounding, each
    within 2^-24 of its value."""
    assert beta_gradient_error(64) < 2.0**-23
