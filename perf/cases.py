"""The attention calls this package is measured on, as a user's program makes them.

Every case goes through torch.nn.functional.scaled_dot_product_attention with
cmpext3's patch in place, the way a program that imports cmpext3 reaches the
kernels; the training cases run the forward and the backward through autograd.
Kernel selection by trial (CMPEXT3_AUTOSELECT) is off: a trial times stock
torch beside the kernel, which is not the work measured here.
"""
from __future__ import annotations

import math
import os
import sys

os.environ["CMPEXT3_AUTOSELECT"] = "0"
sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "torch-cmp-patch_amd"))

import torch  # noqa: E402
import torch.nn.functional as F  # noqa: E402

import cmpext3  # noqa: E402

cmpext3.enable()
cmpext3.enable_backward()

_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}

# Keys of a case
#   dtype, B, H, Hkv (K/V heads, grouped-query when fewer than H), Sq, Sk, D, causal
#   mask    ""      none
#           "pad"   bool [B, 1, 1, Sk], the keys of a padded batch
#           "full"  bool [B, 1, Sq, Sk], causal and left padding in one mask
#   layout  "bshd"  [B, H, S, D] views of [B, S, H, D] memory, what a projection leaves
#           "cache" K and V are the filled part of a longer [B, Hkv, capacity, D] cache
#   train   forward and backward
#   kv_std  standard deviation of K and V


def _case(name, dtype, B, H, Hkv, Sq, Sk, D, causal=False, mask="", layout="bshd", train=False, kv_std=1.0):
    c = dict(dtype=dtype, B=B, H=H, Hkv=Hkv, Sq=Sq, Sk=Sk, D=D, causal=causal, mask=mask, layout=layout,
             train=train, kv_std=kv_std)
    return dict(c, name=name) if name else c


def listed():
    return [
        # the smallest calls: a text encoder's layer over one prompt of 77 tokens
        _case("text_encoder_fp16", "fp16", 1, 12, 12, 77, 77, 64, causal=True),
        # image model, cross-attention to the 77 text tokens, guidance pair
        _case("sdxl_cross_fp16", "fp16", 2, 10, 10, 4096, 77, 64, kv_std=0.5),
        # image model, self-attention over a 64 x 64 latent
        _case("sdxl_self_fp16", "fp16", 2, 10, 10, 4096, 4096, 64),
        # language model, prompts of one length
        _case("qwen3_prefill_bf16", "bf16", 4, 16, 8, 2048, 2048, 128, causal=True),
        # language model, a left-padded batch of prompts of a ragged length
        _case("padded_prefill_bf16", "bf16", 4, 16, 8, 1531, 1531, 128, mask="full"),
        # language model, one token for each of 16 sequences, caches equally full
        _case("qwen3_decode_bf16", "bf16", 16, 16, 8, 1, 4096, 128, layout="cache"),
        # the same of a padded batch, whose step carries the padding mask
        _case("padded_decode_bf16", "bf16", 8, 32, 8, 1, 3001, 128, mask="pad", layout="cache"),
        # full precision: image model, self-attention at head dim 40
        _case("sd15_self_fp32", "fp32", 2, 8, 8, 4096, 4096, 40),
        # full precision, a small training step
        _case("small_train_fp32", "fp32", 1, 8, 8, 1024, 1024, 64, train=True),
        # fine-tuning an image model's self-attention layer
        _case("sdxl_train_fp16", "fp16", 2, 10, 10, 4096, 4096, 64, train=True),
        # training a language model's attention layer
        _case("qwen3_train_bf16", "bf16", 4, 16, 8, 2048, 2048, 128, causal=True, train=True),
        # the largest: training on one long sequence at head dim 256
        _case("long_train_d256_bf16", "bf16", 1, 16, 8, 8192, 8192, 256, causal=True, train=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _drawn(rng):
    kind = rng.choice(["encoder", "cross", "self", "prefill", "padded", "decode", "decode_padded", "fp32",
                       "train_self", "train_causal", "train_fp32"])
    half = rng.choice(["fp16", "bf16"])
    if kind == "encoder":
        s = _log_int(rng, 16, 512)
        return _case("", half, rng.randint(1, 4), rng.choice([8, 12, 16]), 0, s, s, 64, causal=rng.random() < 0.5)
    if kind == "cross":
        return _case("", half, rng.choice([1, 2, 4]), rng.choice([8, 10, 20]), 0, _log_int(rng, 256, 9216),
                     rng.choice([77, rng.randint(32, 128), 154]), rng.choice([40, 64, 80]), kv_std=0.5)
    if kind == "self":
        s = _log_int(rng, 256, 6144)
        return _case("", half, rng.choice([1, 2, 4]), rng.choice([8, 10, 16, 20]), 0, s, s,
                     rng.choice([40, 64, 80, 128, 160]))
    if kind in ("prefill", "padded"):
        s = _log_int(rng, 64, 8192 if kind == "prefill" else 3072)
        h = rng.choice([16, 28, 32])
        return _case("", "bf16" if rng.random() < 0.8 else "fp16", rng.randint(1, 4), h,
                     4 if h == 28 else rng.choice([h, 8]), s, s, rng.choice([64, 128, 128, 256]),
                     causal=kind == "prefill", mask="" if kind == "prefill" else "full")
    if kind in ("decode", "decode_padded"):
        h = rng.choice([16, 28, 32])
        b = rng.choice([1, 2, 8, 16, 32])
        return _case("", "bf16" if rng.random() < 0.8 else "fp16", b, h, 4 if h == 28 else rng.choice([h, 8]),
                     1, _log_int(rng, 128, 262144 // b if b > 8 else 32768), rng.choice([64, 128, 128, 256]),
                     mask="pad" if kind == "decode_padded" else "", layout="cache")
    if kind == "fp32":
        s = _log_int(rng, 77, 4096)
        return _case("", "fp32", rng.choice([1, 2]), rng.choice([8, 10, 12]), 0, s, s, rng.choice([40, 64, 80, 128]),
                     causal=rng.random() < 0.25)
    if kind == "train_self":
        s = _log_int(rng, 256, 5120)
        return _case("", half, rng.choice([1, 2, 4]), rng.choice([8, 10, 16]), 0, s, s, rng.choice([40, 64, 80]),
                     train=True)
    if kind == "train_causal":
        s = _log_int(rng, 128, 4096)
        h = rng.choice([16, 28, 32])
        return _case("", "bf16" if rng.random() < 0.8 else "fp16", rng.randint(1, 4), h,
                     4 if h == 28 else rng.choice([h, 8]), s, s, rng.choice([64, 128, 128, 256]), causal=True,
                     train=True)
    s = _log_int(rng, 77, 1536)
    return _case("", "fp32", rng.choice([1, 2]), rng.choice([8, 12]), 0, s, s, rng.choice([40, 64, 128]),
                 causal=rng.random() < 0.5, train=True)


def draw(rng):
    """One more call of the listed kinds, no dearer than the dearest listed one."""
    most = max(_cost(c) for c in listed())
    while True:
        c = _drawn(rng)
        c["Hkv"] = c["Hkv"] or c["H"]
        if _cost(c) <= most:
            return c


def _pads(case):
    """Keys at the front of each sequence that are padding: none for the
    first sequence, up to half of the keys for the others."""
    return [b * case["Sk"] // (2 * case["B"]) for b in range(case["B"])]


def _mask(case):
    if not case["mask"]:
        return None
    Sq, Sk = case["Sq"], case["Sk"]
    pads = torch.tensor(_pads(case), device="cuda").view(-1, 1, 1, 1)
    key = torch.arange(Sk, device="cuda").view(1, 1, 1, Sk)
    if case["mask"] == "pad":
        return key >= pads
    row = torch.arange(Sq, device="cuda").view(1, 1, Sq, 1)
    # a padding row keeps its own key, so that no row is empty
    return ((key >= pads) & (key <= row)) | (key == row)


def _pairs(case):
    """(query, key) pairs that enter the softmax, over the batch, per head."""
    B, Sq, Sk = case["B"], case["Sq"], case["Sk"]
    if case["mask"] == "pad":
        return sum(Sq * (Sk - p) for p in _pads(case))
    if case["mask"] == "full":
        return sum((Sk - p) * (Sk - p + 1) // 2 + p for p in _pads(case))
    return B * (Sk * (Sk + 1) // 2 if case["causal"] else Sq * Sk)


def work(case):
    es = 4 if case["dtype"] == "fp32" else 2
    B, H, Hkv, Sq, Sk, D = (case[k] for k in ("B", "H", "Hkv", "Sq", "Sk", "D"))
    q, kv = es * B * H * Sq * D, es * B * Hkv * Sk * D
    kept = B * Sk
    if case["mask"] == "pad":  # padding keys need not be read
        kept = sum(Sk - p for p in _pads(case))
    mask = {"": 0, "pad": B * Sk, "full": B * Sq * Sk}[case["mask"]]
    flops = 4 * H * _pairs(case) * D
    if not case["train"]:
        return {"bytes": 2 * q + 2 * kv * kept // (B * Sk) + mask, "flops": flops}
    # forward: q, k, v in, out out.  Backward: q, k, v, out, dout in, dq, dk, dv out, five products for two
    return {"bytes": 2 * q + 2 * kv + 4 * q + 4 * kv, "flops": 3.5 * flops}


def _cost(case):
    w = work(case)
    return w["bytes"] / 5e12 + w["flops"] / (8e13 if case["dtype"] == "fp32" else 6e14)


def _randn(gen, case, heads, S, std=1.0):
    B, D = case["B"], case["D"]
    x = torch.randn(B, S, heads, D, generator=gen, device="cuda") * std
    return x.to(_DTYPES[case["dtype"]]).transpose(1, 2)


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    q = _randn(gen, case, case["H"], case["Sq"])
    k, v = (_randn(gen, case, case["Hkv"], case["Sk"], case["kv_std"]) for _ in range(2))
    if case["layout"] == "cache":
        capacity = (case["Sk"] + 256) // 256 * 256
        full = torch.zeros(2, case["B"], case["Hkv"], capacity, case["D"], dtype=q.dtype, device="cuda")
        for i, x in enumerate((k, v)):
            full[i, :, :, :case["Sk"]] = x
        k, v = (full[i, :, :, :case["Sk"]] for i in range(2))
    state = {"q": q, "k": k, "v": v, "kw": {"attn_mask": _mask(case), "is_causal": case["causal"]}}
    if case["Hkv"] != case["H"]:
        state["kw"]["enable_gqa"] = True
    if case["train"]:
        state["dout"] = _randn(gen, case, case["H"], case["Sq"])
        for name in ("q", "k", "v"):
            state[name].requires_grad_(True)
    return state


def run(state):
    q, k, v = state["q"], state["k"], state["v"]
    out = F.scaled_dot_product_attention(q, k, v, **state["kw"])
    if "dout" not in state:
        return out
    dq, dk, dv = torch.autograd.grad(out, (q, k, v), state["dout"])
    return {"out": out, "dq": dq, "dk": dk, "dv": dv}


def tolerance(case):
    """About four times the largest distance from exact() measured over the
    listed cases and 16 drawn ones.  rel: fp32 1.2e-6, fp16 4.2e-4, bf16
    2.6e-3.  max: fp32 1e-5, fp16 8.2e-3, bf16 0.14 (gradients of the first
    rows of a causal sequence, whose few probabilities are rounded to bf16)."""
    if case["dtype"] == "fp32":
        return {"rel": 5e-6, "max": 4e-5}
    if case["dtype"] == "fp16":
        return {"rel": 1.6e-3, "max": 3.5e-2}
    return {"rel": 1e-2, "max": 5e-1}


def exact(case, seed):
    """The same attention and gradients in float64, one query head at a time."""
    state = prepare(case, seed)
    q, k, v = (state[n].detach() for n in ("q", "k", "v"))
    mask, group = state["kw"]["attn_mask"], case["H"] // case["Hkv"]
    Sq, Sk, scale = case["Sq"], case["Sk"], 1 / math.sqrt(case["D"])
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    train = case["train"]
    if train:
        dq = torch.empty_like(out)
        dk, dv = (torch.zeros(k.shape, dtype=torch.float64, device="cuda") for _ in range(2))
    block = max(1, min(Sq, (1 << 27) // Sk))  # query rows at a time
    for b in range(case["B"]):
        for h in range(case["H"]):
            kd, vd = (t[b, h // group].double().contiguous() for t in (k, v))
            for r in range(0, Sq, block):
                rows = slice(r, min(Sq, r + block))
                qd = q[b, h, rows].double().contiguous()
                s = (qd @ kd.T).mul_(scale)
                if case["causal"]:
                    i = torch.arange(rows.start, rows.stop, device="cuda").view(-1, 1)
                    s.masked_fill_(torch.arange(Sk, device="cuda").view(1, -1) > i, -math.inf)
                if mask is not None:
                    s.masked_fill_(~(mask[b, 0, rows] if mask.shape[2] > 1 else mask[b, 0]), -math.inf)
                p = torch.softmax(s, -1)
                del s
                o = p @ vd
                out[b, h, rows] = o
                if train:
                    g = state["dout"][b, h, rows].double().contiguous()
                    ds = (g @ vd.T).sub_((g * o).sum(-1, keepdim=True)).mul_(p).mul_(scale)
                    dv[b, h // group] += p.T @ g
                    dq[b, h, rows] = ds @ kd
                    dk[b, h // group] += ds.T @ qd
                    del ds
                del p
    return {"out": out, "dq": dq, "dk": dk, "dv": dv} if train else out
