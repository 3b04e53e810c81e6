"""The gradient sweeps share one launch, except where the dQ sweep runs a wave
per SIMD more by itself and the dK/dV grid fills its rounds: both forms, and
both chunk layouts of the tile loader (whole rows; 64-column strips at D =
192), at ragged lengths, with and without K operands parked in LDS.

Reference: autograd of the same attention in float32 on the same (rounded)
inputs.  Bars: tests/test_gpu_backward.py's for fp16/bf16, relative to the
gradient's largest value; fp32: sums of Sk (or Sq x group) products, each off
by a few 2^-24 of its size, against a reference with the same error: 64 * 2^-24
= 4e-6 of the largest value, times 5 for the spread of 10^6 results.
"""
from __future__ import annotations

import pytest
import torch

from cmpext3 import abi

pytestmark = pytest.mark.gpu

BAR = {torch.float32: 2e-5, torch.float16: 1e-2, torch.bfloat16: 2e-2}
F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


def _reference(q, k, v, do, scale, causal, mask):
    """Per batch and K/V head, so that the scores stay small."""
    outs = [torch.empty_like(t, dtype=torch.float32) for t in (q, k, v)]
    G, Sq, Sk = q.shape[1] // k.shape[1], q.shape[2], k.shape[2]
    dead = torch.zeros(Sq, Sk, dtype=torch.bool, device=q.device)
    if causal:
        dead |= torch.ones_like(dead).triu(1)
    for b in range(q.shape[0]):
        gone = dead if mask is None else dead | ~mask[b, 0]
        for h in range(k.shape[1]):
            qs, ks, vs = (t.detach().float().clone().requires_grad_(True)
                          for t in (q[b, h * G:(h + 1) * G], k[b, h], v[b, h]))
            p = ((qs.reshape(-1, qs.shape[-1]) @ ks.t()).view(G, Sq, Sk) * scale).masked_fill(gone, -torch.inf)
            o = (torch.softmax(p, -1).view(G * Sq, Sk) @ vs).view(G, Sq, -1)
            g = torch.autograd.grad(o, (qs, ks, vs), do[b, h * G:(h + 1) * G].float())
            outs[0][b, h * G:(h + 1) * G], outs[1][b, h], outs[2][b, h] = g
    return outs


@pytest.mark.parametrize("dtype,B,H,Hkv,S,D,causal,masked", [
    (BF16, 2, 16, 16, 2048, 64, True, False),   # 512 key blocks, two a CU
    (F16, 2, 16, 16, 2047, 64, True, True),
    (F16, 2, 32, 16, 2047, 64, True, True),     # and 1024 query blocks, masked: a launch each
    (BF16, 4, 16, 16, 1000, 64, True, True),    # 512 and 512: one launch
    (BF16, 2, 15, 15, 2048, 64, True, False),
    (F16, 2, 6, 3, 333, 64, False, True),       # K operands parked
    (F32, 2, 8, 8, 2040, 40, False, False),     # 512 key blocks: a launch each
    (F32, 2, 8, 8, 1890, 40, False, False),     # 480: one launch
    (F32, 2, 8, 8, 2040, 32, True, False),
    (BF16, 2, 4, 2, 333, 128, True, False),     # K operands parked
    (F16, 1, 4, 4, 333, 120, False, True),
    (BF16, 1, 4, 4, 257, 128, True, True),
    (F16, 1, 4, 2, 520, 192, True, False),      # 64-column strips
    (BF16, 1, 3, 3, 161, 136, False, True),     # and columns past D
    (BF16, 1, 2, 2, 300, 256, True, True),
])
def test_backward_launches(dtype, B, H, Hkv, S, D, causal, masked):
    g = torch.Generator(device="cuda").manual_seed(S * 7 + D)
    q, do = (torch.randn(B, H, S, D, generator=g, device="cuda").to(dtype) for _ in range(2))
    k, v = (torch.randn(B, Hkv, S, D, generator=g, device="cuda").to(dtype) for _ in range(2))
    mask = None
    if masked:  # padding at the end; key 0 stays
        mask = torch.arange(S, device="cuda").view(1, 1, 1, S) < S - S // 5
        mask = mask.expand(B, 1, S, S).contiguous()
    scale = D ** -0.5
    out, lse = abi.attn_fwd_lse(q, k, v, scale, causal, attn_mask=mask)
    delta = torch.empty(B, H, S, device="cuda")
    want = _reference(q, k, v, do, scale, causal, mask)
    for workspace in (None, True):  # whole and split sweeps
        got = [torch.full_like(t, torch.nan) for t in (q, k, v)]
        assert abi.attn_bwd_raw(q, k, v, out, do, lse, *got, delta, scale, causal, attn_mask=mask,
                                workspace=workspace) == 0
        for name, a, b in zip(("dq", "dk", "dv"), got, want):
            err = float((a.float() - b).abs().max() / b.abs().max())
            assert err <= BAR[dtype], (name, err)
