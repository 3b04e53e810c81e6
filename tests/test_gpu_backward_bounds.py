"""GPU check that the training pair reads nothing past a head's last row.

q, k, v and dout are heads inside larger allocations whose other rows (behind
every head, the last one included) hold NaN.  A row read from there reaches
dK, dV or dQ as 0 * NaN, so finite, correct gradients show that the tail of a
ragged last tile reads zeros.  Gradients against the float64 oracle, relative
to each gradient's largest value (bar: 1e-2 fp16, 2e-2 bf16, 1e-4 fp32).
"""
from __future__ import annotations

import pytest
import torch

from cmpext3 import abi
from oracle import sdpa_oracle as orc

pytestmark = pytest.mark.gpu

TOL = orc.TOLERANCE
TDT = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}


def _heads(g, dtype, B, H, S, D, bshd):
    """[B, H, S, D] of N(0, 1) whose neighbouring rows in memory are NaN."""
    x = torch.randn(B, H, S, D, generator=g).to(TDT[dtype])
    if bshd:
        buf = torch.full((B, S + 70, H, D), float("nan"), dtype=x.dtype, device="cuda")
        view = buf[:, :S].transpose(1, 2)
    else:
        buf = torch.full((B, H, S + 70, D), float("nan"), dtype=x.dtype, device="cuda")
        view = buf[:, :, :S]
    view.copy_(x)
    return view


CASES = [(dt, B, H, Hkv, S, S, D, causal, bshd)
         for dt, B, H, Hkv in (("bf16", 1, 2, 1), ("fp16", 2, 2, 2))
         for S in (33, 333) for D in (64, 80, 128, 192, 256) for causal, bshd in ((False, False), (True, True))]
CASES += [("bf16", 1, 4, 2, 65, 417, 128, False, False), ("fp32", 1, 2, 2, 333, 333, 64, True, False),
          ("fp32", 1, 2, 1, 33, 33, 128, False, True)]


@pytest.mark.parametrize("case", CASES, ids=["-".join(map(str, c)) for c in CASES])
def test_rows_past_a_head_are_not_read(case):
    dtype, B, H, Hkv, Sq, Sk, D, causal, bshd = case
    print(f"bounds {case}", flush=True)
    g = torch.Generator().manual_seed(Sq + D)
    q, do = (_heads(g, dtype, B, H, Sq, D, bshd) for _ in range(2))
    k, v = (_heads(g, dtype, B, Hkv, Sk, D, bshd) for _ in range(2))
    out, lse = abi.attn_fwd_lse(q, k, v, D ** -0.5, causal)
    rep = lambda t: t.cpu().repeat_interleave(H // Hkv, dim=1)
    assert orc.max_abs_err(out.cpu(), orc.sdpa_np(q.cpu(), rep(k), rep(v), D ** -0.5, causal)) <= TOL[dtype]
    want = [torch.as_tensor(t) for t in orc.sdpa_bwd_np(q.cpu(), rep(k), rep(v), do.cpu(), D ** -0.5, causal)]
    want[1:] = [t.view(B, Hkv, H // Hkv, Sk, D).sum(2) for t in want[1:]]
    for ws in (True, None):  # with split sweeps where the plan has them, and whole
        got = abi.attn_bwd(q, k, v, out, do, lse, D ** -0.5, causal, workspace=ws)
        torch.cuda.synchronize()
        for name, a, b in zip(("dq", "dk", "dv"), got, want):
            a = a.cpu().double()
            assert torch.isfinite(a).all(), name
            assert (a - b).abs().max() <= TOL[dtype] * b.abs().max(), name
