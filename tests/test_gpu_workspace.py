"""GPU checks of the workspace that the torch binding and cmpext3.abi keep per
stream, where bool masks in bit form (up to 128 MiB) go through it.

Prompts of rising length must not each make a new workspace; a mask of more
than 16 MiB of bits takes one for its call alone, which is given back.
"""
from __future__ import annotations

import pytest
import torch

import cmpext3
from cmpext3 import abi

pytestmark = pytest.mark.gpu


def _call(B, H, S, per_head, D=64, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    q, k, v = (torch.randn(B, H, S, D, generator=g, device="cuda").half() for _ in range(3))
    m = torch.rand(B, H if per_head else 1, S, S, generator=g, device="cuda") > 0.4
    m[..., 0] = True
    return q, k, v, m


def test_rising_lengths_share_a_workspace():
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        sizes = []
        for S in range(520, 1500, 60):
            q, k, v, m = _call(2, 4, S, False, seed=S)
            cmpext3.ops.attention(q, k, v, None, False, m)
            sizes.append(cmpext3.ops.workspace_bytes(torch.cuda.current_device()))
    torch.cuda.synchronize()
    assert sizes[0] > 0 and sizes == sorted(sizes)
    # 17 lengths: a new one per 4 MiB of need
    assert len(set(sizes)) <= max(sizes) >> 22 and all(n % (4 << 20) == 0 for n in set(sizes)), set(sizes)


@pytest.mark.parametrize("side", ["binding", "abi", "abi, another stream"])
def test_a_large_masks_workspace_is_given_back(side):
    B, H, S = 1, 20, 2600  # 17 MB of bits
    q, k, v, m = _call(B, H, S, True)
    assert abi.mask_workspace_size(abi.DTYPE_F16, B, H, H, S, S, 64, abi.DTYPE_BOOL, m.stride()[:3]) > 16 << 20
    want = torch.empty_like(q)  # the mask read as it is
    assert abi.attn_fwd_raw(q, k, v, want, 0.125, False, attn_mask=m, workspace=False) == 0
    small = _call(1, 2, 600, False)
    other = torch.cuda.Stream()

    def run(q, k, v, m):
        if side == "binding":
            return cmpext3.ops.attention(q, k, v, None, False, m)
        out = torch.empty_like(q)
        stream = other if side != "abi" else None
        if stream is not None:
            stream.wait_stream(torch.cuda.current_stream())
        assert abi.attn_fwd_raw(q, k, v, out, 0.125, False, attn_mask=m, stream=stream) == 0
        if stream is not None:
            torch.cuda.current_stream().wait_stream(stream)
        return out

    first = run(*small)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    outs = [run(q, k, v, m) for _ in range(3)]
    torch.cuda.synchronize()
    out_bytes = (q.numel() * 2 + 511) // 512 * 512
    assert torch.cuda.memory_allocated() - before == 3 * out_bytes
    assert torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])
    # two sums of the same probabilities (fp16) in another order, 1e-3 of
    # outputs of at most a few units
    assert (outs[0].float() - want.float()).abs().max() <= 4e-3
    assert torch.equal(run(*small), first)
