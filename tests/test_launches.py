"""What reaches a stream when C entry points are called (no GPU).

The library runs against tests/launch_recorder.cpp, which records launches
instead of making them, in a process of its own.  Tensors are addresses that
nothing on the host reads.
"""
from __future__ import annotations

import json
import subprocess
import sys
from pathlib import Path

import pytest

HERE = Path(__file__).resolve().parent
LIB = HERE.parent / "torch-cmp-patch_amd" / "cmpext3" / "libcmpext3_attn.so"

PRELUDE = """
import ctypes, json, sys, threading
rec = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL(sys.argv[2])
vp, ci, sz, i64 = ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t, ctypes.c_int64
lib.cmpext3_attn_bwd_workspace_size.restype = sz
lib.cmpext3_attn_fwd_workspace_size.restype = sz
F16, BF16, F32, BOOL = 0, 1, 2, 3
A = 1 << 32                                     # stands for every tensor
s3 = lambda *s: (i64 * 3)(*s)
def fwd(entry, dt, B, H, S, D, mask, ws=None, nbytes=0, causal=0):
    st = s3(H * S * D, S * D, D)
    ms = s3(0, 0, S) if mask else s3(0, 0, 0)
    tail = [vp(A) if mask else None, BOOL if mask else -1, ms, ctypes.c_float(0.1), causal]
    if entry == "ws":
        tail += [vp(ws), sz(nbytes), None]
        f = lib.cmpext3_attn_fwd_ws
    else:
        tail += [None]
        f = lib.cmpext3_attn_fwd_noalloc
    return f(vp(A), vp(A), vp(A), vp(A), dt, B, H, H, S, S, D, st, st, st, st, *tail)
def bwd(dt, B, H, Hkv, Sq, Sk, D, causal, ws=None, nbytes=0, mask=False):
    q, k = s3(H * Sq * D, Sq * D, D), s3(Hkv * Sk * D, Sk * D, D)
    return lib.cmpext3_attn_bwd_ws(*[vp(A)] * 10, dt, B, H, Hkv, Sq, Sk, D, q, k, k, q, q, q, k, k,
                                   vp(A) if mask else None, BOOL if mask else -1, s3(0, 0, 0), ctypes.c_float(0.1), causal, vp(ws), sz(nbytes), None)
def launches():
    out = []
    for i in range(rec.recorder_count()):
        name, wg, th = ctypes.c_char_p(), ctypes.c_uint64(), ctypes.c_uint64()
        tag = rec.recorder_get(i, ctypes.byref(name), ctypes.byref(wg), ctypes.byref(th))
        out.append((tag, name.value.decode(), wg.value, th.value))
    return out
"""


@pytest.fixture(scope="module")
def recorder(tmp_path_factory):
    so = tmp_path_factory.mktemp("recorder") / "launch_recorder.so"
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", "-pthread", str(HERE / "launch_recorder.cpp"),
                    "-o", str(so)], check=True)
    return so


def _run(recorder, body):
    res = subprocess.run([sys.executable, "-c", PRELUDE + body, str(recorder), str(LIB)], capture_output=True,
                         text=True, timeout=120)
    assert res.returncode == 0, res.stderr
    return json.loads(res.stdout)


# Two threads on one stream with one workspace (or the library's fixed one):
# a bool-masked call makes its mask's bits there and then reads them, so no
# other call's launch may come between the two.
@pytest.mark.parametrize("entry,other", [("ws", "masked"), ("ws", "split"), ("ws", "backward"),
                                         ("noalloc", "masked"), ("noalloc", "split")])
def test_a_masked_calls_launches_stay_together(recorder, entry, other):
    got = _run(recorder, f"""
entry, other = {entry!r}, {other!r}
rec.recorder_slow(b"attn_mask_bits", 3000)
n, ws, done, rcs = 1 << 28, 1 << 34, [], set()
def masked(tag):
    rec.recorder_tag(tag)
    for _ in range(8):
        rcs.add(fwd(entry, BF16, 1, 2, 700, 128, True, ws, n))
    done.append(tag)
def second():
    if other == "masked":
        return masked(2)
    rec.recorder_tag(2)
    while True:
        rcs.add(fwd(entry, BF16, 1, 8, 1024, 128, False, ws, n) if other == "split"
                else bwd(BF16, 1, 8, 2, 1024, 1024, 128, 1, ws, n))
        if done:
            break
ts = [threading.Thread(target=masked, args=(1,)), threading.Thread(target=second)]
[t.start() for t in ts]; [t.join() for t in ts]
print(json.dumps([sorted(rcs), launches()]))
""")
    rcs, seen = got
    assert rcs == [0]
    assert {tag for tag, *_ in seen} == {1, 2}
    bits = [i for i, (_, name, *_) in enumerate(seen) if "attn_mask_bits" in name]
    assert len(bits) == (16 if other == "masked" else 8)
    for i in bits:
        assert seen[i + 1][0] == seen[i][0] and "attn_fwd_pipe16" in seen[i + 1][1], seen[max(0, i - 2):i + 4]


# HIP takes fewer than 2^32 threads per grid.  Many short sequences: each
# gradient sweep's grid is within that, the two together are not.
@pytest.mark.parametrize("dt,D,causal", [("F16", 64, 0), ("BF16", 64, 1), ("BF16", 128, 0), ("F32", 32, 1), ("F32", 40, 0)])
def test_backward_grids_stay_launchable(recorder, dt, D, causal):
    rc, seen = _run(recorder, f"""
rc = bwd({dt}, 3000, 3000, 3000, 1, 1, {D}, {causal})
print(json.dumps([rc, launches()]))
""")
    assert rc == 0
    assert all(threads < 2 ** 32 for *_, threads in seen), seen
    # nothing is lost: a workgroup per block of keys and of queries
    assert sum(wg for _, name, wg, _ in seen if "grads" in name) == 2 * 3000 * 3000


# The gradient sweeps share one launch, except where the dQ sweep runs a wave
# per SIMD more by itself and both grids fill their rounds.
@pytest.mark.parametrize("dt,B,H,Hkv,S,D,causal,mask,n", [
    ("BF16", 4, 16, 8, 2048, 64, 1, True, 2),
    ("BF16", 4, 32, 32, 1024, 64, 1, True, 2),
    ("BF16", 4, 16, 8, 2048, 64, 1, False, 1),     # without a mask
    ("BF16", 2, 16, 16, 2048, 64, 1, True, 1),     # 512 dQ blocks
    ("BF16", 4, 32, 16, 1024, 64, 1, True, 1),     # 512 dK/dV blocks of short sweeps
    ("BF16", 4, 15, 15, 2048, 64, 1, True, 1),     # a partial round
    ("F16", 4, 32, 32, 1024, 64, 0, True, 1),
    ("F32", 2, 8, 8, 3000, 40, 0, False, 2),
    ("F32", 2, 8, 8, 3000, 64, 0, False, 1),
])
def test_backward_launch_forms(recorder, dt, B, H, Hkv, S, D, causal, mask, n):
    rc, seen = _run(recorder, f"""
rc = bwd({dt}, {B}, {H}, {Hkv}, {S}, {S}, {D}, {causal}, mask={mask})
print(json.dumps([rc, launches()]))
""")
    assert rc == 0
    assert sum("grads" in name for _, name, *_ in seen) == n


def test_backward_plans_count_the_one_launch():
    """Three workgroups per CU at D <= 64, masked too (a dQ grid of 128 blocks
    takes six parts); a partial round is cut only where it is the last that
    the CUs have room for (no tails of 384 blocks at three per CU)."""
    import torch
    from cmpext3 import abi
    if torch.cuda.is_available():
        pytest.skip("plan depends on the visible device's CU count")
    size = lambda B, H, S, mask: abi.bwd_workspace_size(abi.DTYPE_F16, B, H, H, S, S, 64, mask, False)
    assert size(1, 8, 2048, abi.DTYPE_BOOL) == (2 * 6 + 6) * 8 * 2048 * 64 * 4
    assert size(4, 16, 700, -1) == 0


def test_mask_workspace_is_asked_for_by_launches_that_fill_it(recorder):
    """The size query against the launches: bytes exactly where a call with room
    for them makes the bits (element-wise masks: Sk not a multiple of 8)."""
    got = _run(recorder, """
lib.cmpext3_attn_fwd_mask_workspace_size.restype = sz
out = []
for dt in (F16, BF16, F32):
    for B, H, S in ((1, 4, 1), (2, 4, 20), (2, 4, 77), (4, 16, 203), (1, 8, 517), (2, 8, 2045)):
        for D in (32, 44, 64, 80, 100, 128, 160, 192, 256):
            for causal in (0, 1):
                rec.recorder_clear()
                size = lib.cmpext3_attn_fwd_mask_workspace_size(dt, B, H, H, S, S, D, BOOL, s3(0, 0, S), causal)
                if dt == F32 and D % 4:
                    continue
                rc = fwd("ws", dt, B, H, S, D, True, 1 << 34, 1 << 30, causal)
                out.append([dt, B, H, S, D, causal, rc, size, sum("attn_mask_bits" in n for _, n, *_ in launches())])
print(json.dumps(out))
""")
    assert len(got) > 300 and any(size for *_, size, _ in got)
    for *case, rc, size, made in got:
        assert rc == 0 and (size > 0) == (made == 1), (case, size, made)


@pytest.mark.parametrize("H,S,D,parts", [
    (2, 1024, 64, 2), (2, 2048, 64, 4), (2, 2048, 256, 4), (4, 2048, 128, 4), (6, 2048, 64, 3),
    (8, 2048, 64, 3), (8, 3072, 64, 3), (2, 6000, 64, 4), (12, 2048, 64, 2), (16, 2048, 64, 2),
    (32, 1024, 128, 1)])
def test_small_causal_grids_keep_a_part_per_cu(H, S, D, parts):
    import torch
    from cmpext3 import abi
    if torch.cuda.is_available():
        pytest.skip("plan depends on the visible device's CU count")
    assert abi.plan(abi.DTYPE_BF16, 1, H, H, S, S, D, 1 << 40, causal=True) == (abi.OK, parts)
