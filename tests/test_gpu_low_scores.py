"""GPU parity where every score of a row is far below zero.

A row's first live key sets the exponentials' offset.  From 128 below it in
the exp2 domain (a scaled score of -88.7) 2^-offset overflows, and a kernel
that scales its still empty sums by it turns the row into NaN.  Scores get
there with opposed Q and K (here near -128), and with additive masks that add
a large negative number to dropped keys: an all -65504 first tile.  Cases:
every kernel that keeps a running offset, unsplit, in two and in more parts
(each part sets its own offset), masks of every kind, the training forward.
Checked against the float64 oracle (bar: max abs error 1e-2 fp16, 2e-2 bf16,
1e-4 fp32).
"""
from __future__ import annotations

import pytest
import torch

from cmpext3 import abi
from oracle import sdpa_oracle as orc

pytestmark = pytest.mark.gpu

TOL = orc.TOLERANCE
TDT = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _low(dtype, B, H, Sq, Sk, D):
    """Q = 4, K near -4, scale so that every score is near -128 (-185 in the
    exp2 domain); V normal."""
    g = torch.Generator().manual_seed(Sk + D)
    q = torch.full((B, H, Sq, D), 4.0)
    k = torch.randn(B, H, Sk, D, generator=g) * 0.125 - 4.0
    v = torch.randn(B, H, Sk, D, generator=g)
    return *(x.to(TDT[dtype]).cuda() for x in (q, k, v)), 128.0 / (16 * D)


LOW = [
    # dtype, B, H, Sq, Sk, D, causal, key parts (1: no workspace, 3: or more)
    ("fp16", 1, 2, 300, 1000, 64, False, 1),
    ("bf16", 1, 2, 300, 1000, 128, False, 1),
    ("bf16", 1, 8, 1024, 1024, 128, False, 2),
    ("fp16", 1, 8, 1024, 1024, 64, True, 2),
    ("bf16", 1, 2, 300, 1000, 128, False, 3),
    ("fp16", 1, 2, 200, 2600, 80, False, 3),
    ("bf16", 1, 2, 300, 700, 256, False, 1),
    ("fp16", 1, 2, 200, 200, 160, True, 1),     # head-dim > 128 kernel
    ("bf16", 1, 2, 40, 900, 192, False, 1),
    ("fp16", 1, 2, 100, 77, 64, False, 1),      # short-key kernel
    ("bf16", 1, 2, 1, 3000, 128, False, 3),     # decode kernel
    ("fp32", 1, 2, 200, 700, 40, True, 1),
]


@pytest.mark.parametrize("case", LOW, ids=["-".join(map(str, c)) for c in LOW])
def test_low_scores(case):
    dtype, B, H, Sq, Sk, D, causal, parts = case
    print(f"low scores {case}", flush=True)
    q, k, v, scale = _low(dtype, B, H, Sq, Sk, D)
    if parts > 1:
        got = abi.plan(abi.dtype_code(TDT[dtype]), B, H, H, Sq, Sk, D, 1 << 40, causal=causal)[1]
        assert got == 2 if parts == 2 else got >= 3
    out = torch.full_like(q, float("nan"))
    assert abi.attn_fwd_raw(q, k, v, out, scale, causal, workspace=parts > 1) == 0
    torch.cuda.synchronize()
    want = orc.sdpa_np(q.cpu(), k.cpu(), v.cpu(), scale, causal)
    assert orc.max_abs_err(out.cpu(), want) <= TOL[dtype]


@pytest.mark.parametrize("dtype,Sk,D", [("fp16", 1000, 64), ("bf16", 1000, 128), ("bf16", 1001, 128), ("fp16", 700, 256)])
@pytest.mark.parametrize("workspace", [True, False])
def test_low_scores_bool_mask(dtype, Sk, D, workspace):
    """In bit form (with room for it) and read as it is."""
    q, k, v, scale = _low(dtype, 2, 2, 300, Sk, D)
    g = torch.Generator().manual_seed(Sk)
    keep = torch.rand(2, 1, 300, Sk, generator=g) > 0.5
    keep[1, :, :, :200] = False
    out = torch.full_like(q, float("nan"))
    assert abi.attn_fwd_raw(q, k, v, out, scale, False, attn_mask=keep.cuda(), workspace=workspace) == 0
    torch.cuda.synchronize()
    want = orc.sdpa_np(q.cpu(), k.cpu(), v.cpu(), scale, False, attn_mask=keep)
    assert orc.max_abs_err(out.cpu(), want) <= TOL[dtype]


LEAST = [
    # dtype, mask dtype, Sq, Sk, D, mask rows
    ("fp16", "fp16", 300, 1000, 64, 1),
    ("fp16", "fp16", 300, 1000, 64, 300),
    ("bf16", "fp16", 300, 1001, 128, 300),      # read element by element
    ("bf16", "fp16", 300, 700, 256, 300),
    ("fp16", "fp16", 40, 200, 160, 1),          # head-dim > 128 kernel
    ("bf16", "bf16", 300, 1000, 128, 1),
    ("fp16", "fp32", 300, 1000, 64, 1),
    ("bf16", "fp16", 1, 3001, 128, 1),          # decode kernel
    ("fp32", "fp16", 200, 700, 64, 1),
]


@pytest.mark.parametrize("case", LEAST, ids=["-".join(map(str, c)) for c in LEAST])
@pytest.mark.parametrize("workspace", [True, False])
def test_lowest_value_masks(case, workspace):
    """Left padding as an additive mask of the type's lowest value: its first
    keys (more than a tile) are all dropped, each row keeps later ones."""
    dtype, mdt, Sq, Sk, D, rows = case
    print(f"lowest value {case} {workspace}", flush=True)
    g = torch.Generator().manual_seed(Sk)
    q, k, v = (torch.randn(2, 2, s, D, generator=g).to(TDT[dtype]).cuda() for s in (Sq, Sk, Sk))
    m = torch.zeros(2, 1, rows, Sk, dtype=TDT[mdt])
    m[0, ..., :40] = torch.finfo(TDT[mdt]).min
    m[1, ..., :Sk // 2] = torch.finfo(TDT[mdt]).min
    out = torch.full_like(q, float("nan"))
    assert abi.attn_fwd_raw(q, k, v, out, D ** -0.5, False, attn_mask=m.cuda(), workspace=workspace) == 0
    torch.cuda.synchronize()
    want = orc.sdpa_np(q.cpu(), k.cpu(), v.cpu(), D ** -0.5, False, attn_mask=m)
    assert orc.max_abs_err(out.cpu(), want) <= TOL[dtype]


@pytest.mark.parametrize("dtype,Sq,Sk,D,causal", [("fp16", 300, 1000, 64, False), ("bf16", 512, 512, 128, True),
                                                  ("bf16", 300, 700, 256, False), ("bf16", 40, 200, 192, True)])
def test_low_scores_training_forward(dtype, Sq, Sk, D, causal):
    q, k, v, scale = _low(dtype, 1, 2, Sq, Sk, D)
    out, lse = abi.attn_fwd_lse(q, k, v, scale, causal)
    torch.cuda.synchronize()
    want = orc.sdpa_np(q.cpu(), k.cpu(), v.cpu(), scale, causal)
    assert orc.max_abs_err(out.cpu(), want) <= TOL[dtype]
    # scores near -128; fp16 Q pre-scaled into fp16: 2^-11 of them, half an ulp each way
    ref = torch.as_tensor(orc.sdpa_lse_np(q.cpu(), k.cpu(), scale, causal)).reshape(lse.shape)
    assert (lse.cpu().double() - ref).abs().max() <= 128 * 2.0 ** -11 + 1e-3
