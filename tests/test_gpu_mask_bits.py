"""GPU parity of bool masks in bit form (attn_fwd_mask_bits.hip and the
pipelined kernel's OPT bit 11).

A non-causal f16/bf16 launch with a bool mask and room in its workspace first
turns the mask into one word per row and 32-key tile and a class per 128-row
block and tile, and its sweep then leaves out the tiles a block keeps no pair
of.  Checked against the float64 oracle (bar: max abs error 1e-2 fp16, 2e-2
bf16), against a rerun (bit-identical) and against the same call without a
workspace, which reads the mask as it is.
"""
from __future__ import annotations

import pytest
import torch

import cmpext3
from cmpext3 import abi
from cmpext3 import workloads as W
from oracle import sdpa_oracle as orc

TOL = orc.TOLERANCE
TDT = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _mask(kind, B, H, Sq, Sk, seed):
    g = torch.Generator().manual_seed(seed)
    row = torch.arange(Sq).view(1, 1, Sq, 1)
    key = torch.arange(Sk).view(1, 1, 1, Sk)
    pad = torch.tensor([b * Sk // (2 * B) + 3 * (b > 0) for b in range(B)]).view(B, 1, 1, 1)
    if kind == "left_pad":                     # causal and left padding, one mask for all heads
        return (key <= row) & (key >= pad)     # rows of the padding see nothing
    if kind == "random_heads":                 # per head, most pairs dropped, one block without any
        m = torch.rand(B, H, Sq, Sk, generator=g) > 0.9
        m[0, 0, 128:256] = False
        return m
    if kind == "band":                         # a few tiles of a long sweep: fewer than the key split's parts
        m = (key >= 40) & (key < 70) & (row >= 0)
        return m.expand(1, 1, Sq, Sk).clone()
    if kind == "keys":                         # one row for all queries
        m = (key >= pad) & (key % 97 != 5)
        m[..., 64:128] = True                  # tiles that need no mask
        return m
    if kind == "all":                          # nothing dropped
        return torch.ones(1, 1, Sq, Sk, dtype=torch.bool)
    assert kind == "view"                      # rows of a wider buffer, one byte off, bytes other than 0 and 1
    buf = torch.randint(0, 4, (B, Sq, Sk + 7), generator=g, dtype=torch.uint8) * 85
    return buf.cuda().view(torch.bool)[..., 1:Sk + 1][:, None]


CASES = [
    # dtype, B, H, Hkv, Sq, Sk, D, mask, scale
    ("bf16", 3, 4, 2, 333, 333, 128, "left_pad", None),
    ("fp16", 2, 4, 4, 700, 700, 64, "left_pad", None),
    ("fp16", 1, 3, 3, 300, 1000, 32, "random_heads", None),
    ("bf16", 1, 2, 1, 300, 777, 40, "random_heads", None),
    ("fp16", 1, 2, 2, 256, 2048, 80, "band", None),
    ("bf16", 1, 2, 2, 130, 5000, 128, "keys", None),       # list windows past 64 and 128 tiles
    ("fp16", 2, 2, 2, 200, 2600, 64, "keys", 1.5),         # Q not pre-scaled
    ("bf16", 2, 2, 2, 257, 290, 96, "all", None),
    ("fp16", 1, 2, 2, 100, 4500, 64, "all", None),
    ("fp16", 2, 2, 2, 150, 515, 96, "view", -0.2),
    ("bf16", 1, 2, 2, 129, 256, 64, "view", 0.0),
    ("bf16", 2, 4, 2, 400, 400, 256, "left_pad", None),    # one wave per SIMD
    ("fp16", 1, 2, 2, 280, 600, 160, "random_heads", None),
    ("bf16", 1, 2, 2, 280, 600, 192, "view", None),
]


@pytest.mark.gpu
@pytest.mark.parametrize("case", CASES, ids=[f"{c[0]}-b{c[1]}h{c[2]}of{c[3]}-q{c[4]}k{c[5]}d{c[6]}-{c[7]}" for c in CASES])
def test_bool_mask_in_bit_form(case):
    dtype, B, H, Hkv, Sq, Sk, D, kind, scale = case
    print(f"mask bits {case}", flush=True)
    q = W.Workload("bq", dtype, B, H, Sq, Sk, D, seed=Sq).make_inputs("cuda")[0]
    _, k, v = W.Workload("bk", dtype, B, Hkv, Sq, Sk, D, seed=Sk).make_inputs("cuda")
    scale = D ** -0.5 if scale is None else scale
    m = _mask(kind, B, H, Sq, Sk, seed=D).cuda()
    em = m.expand(B, H, Sq, Sk)
    assert abi.mask_workspace_size(abi.dtype_code(TDT[dtype]), B, H, Hkv, Sq, Sk, D, abi.DTYPE_BOOL,
                                   em.stride()[:3]) > 0
    outs = [torch.full_like(q, float("nan")) for _ in range(3)]
    for out, ws in zip(outs, (True, True, False)):
        assert abi.attn_fwd_raw(q, k, v, out, scale, False, attn_mask=m, workspace=ws) == 0
    torch.cuda.synchronize()
    g = H // Hkv
    keep = (m.view(torch.uint8) != 0).cpu()
    want = orc.sdpa_np(q.cpu(), k.cpu().repeat_interleave(g, dim=1), v.cpu().repeat_interleave(g, dim=1), scale,
                       False, attn_mask=keep)
    assert torch.equal(outs[0], outs[1])
    for out in (outs[0], outs[2]):
        assert orc.max_abs_err(out.cpu(), want) <= TOL[dtype]
    dead = ~keep.expand(B, H, Sq, Sk).any(-1)
    assert not outs[0].cpu()[dead].any()


@pytest.mark.gpu
def test_allocation_free_entry_point_makes_the_bits_too():
    q, k, v = W.Workload("bn", "fp16", 2, 4, 300, 900, 64, seed=3).make_inputs("cuda")
    m = _mask("random_heads", 2, 4, 300, 900, seed=1).cuda()
    ws = torch.zeros(abi.NOALLOC_SCRATCH_BYTES, dtype=torch.uint8, device="cuda")
    a, b = torch.empty_like(q), torch.empty_like(q)
    assert abi.attn_fwd_noalloc_raw(q, k, v, a, 0.125, attn_mask=m) == 0
    assert abi.attn_fwd_raw(q, k, v, b, 0.125, attn_mask=m, workspace=ws) == 0
    torch.cuda.synchronize()
    assert torch.equal(a, b)


def _tell_tale(dtype, Sq, Sk, D):
    """Inputs whose result says whether the bits were made: V is NaN over key
    tiles that no query keeps.  The bit form leaves those tiles out; the mask
    read as it is weighs them 0, and 0 * NaN is NaN."""
    q, k, v = W.Workload("bt", dtype, 2, 4, Sq, Sk, D, seed=Sk).make_inputs("cuda")
    m = _mask("left_pad", 2, 4, Sq, Sk, 0) & (torch.arange(Sk) // 32 != 2)
    m |= torch.arange(Sk) < 8  # every row keeps a key
    nan = v.clone()
    nan[:, :, 64:96] = float("nan")
    keep = m.expand(2, 4, Sq, Sk)
    return q, k, nan, m.cuda(), orc.sdpa_np(q.cpu(), k.cpu(), v.cpu(), D ** -0.5, False, attn_mask=keep)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,Sq,Sk,D", [("fp16", 300, 777, 64), ("bf16", 300, 776, 128), ("bf16", 520, 1001, 128),
                                           ("fp16", 300, 600, 192)])
@pytest.mark.parametrize("side", ["abi", "given workspace", "allocation-free", "binding"])
def test_the_bits_are_made(dtype, Sq, Sk, D, side):
    q, k, v, m, want = _tell_tale(dtype, Sq, Sk, D)
    out = torch.empty_like(q)
    if side == "abi":
        assert abi.attn_fwd_raw(q, k, v, out, D ** -0.5, False, attn_mask=m) == 0
    elif side == "given workspace":
        ws = torch.zeros(16 << 20, dtype=torch.uint8, device="cuda")
        assert abi.attn_fwd_raw(q, k, v, out, D ** -0.5, False, attn_mask=m, workspace=ws) == 0
    elif side == "allocation-free":
        assert abi.attn_fwd_noalloc_raw(q, k, v, out, D ** -0.5, False, attn_mask=m) == 0
    else:
        out = cmpext3.ops.attention(q, k, v, None, False, m)
    as_it_is = torch.empty_like(q)
    assert abi.attn_fwd_raw(q, k, v, as_it_is, D ** -0.5, False, attn_mask=m, workspace=False) == 0
    torch.cuda.synchronize()
    assert torch.isfinite(out).all() and orc.max_abs_err(out.cpu(), want) <= TOL[dtype]
    assert torch.isnan(as_it_is).any()  # the inputs do tell the two apart


def test_mask_workspace_size():
    """One bit per mask element, dimensions broadcast over once, plus a byte
    per 128 rows x 32 keys; nothing for launches that read no bits."""
    size = lambda **kw: abi.mask_workspace_size(*(kw.get(n, d) for n, d in [
        ("dt", abi.DTYPE_BF16), ("B", 4), ("H", 16), ("Hkv", 8), ("Sq", 1531), ("Sk", 1531), ("D", 128),
        ("mdt", abi.DTYPE_BOOL), ("st", (1531 * 1531, 0, 1531))]), kw.get("causal", False))
    up = lambda n: (n + 255) // 256 * 256
    assert size() == up(4 * 48 * 1531 * 4) + up(4 * 12 * 48) + 256
    assert size(st=(0, 0, 1531)) == up(48 * 1531 * 4) + up(12 * 48) + 256
    assert size(st=(1531, 0, 0)) == up(4 * 48 * 4) + up(4 * 48) + 256
    assert size(causal=True) == size(mdt=abi.DTYPE_F16) == size(dt=abi.DTYPE_F32) == size(Sk=31) == 0
    assert size(Sq=1) == 0                              # the decode kernel's
    assert size(Sk=65537) == 0                          # more tiles than a block's list holds
    assert size(Sq=40000, Sk=40000, st=(1, 1, 1)) == 0  # past the size kept for it
    assert size(D=300) == 0
