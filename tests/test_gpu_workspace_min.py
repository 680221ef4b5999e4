"""Calls with less scratch than their fastest kernels take: the least workspace
of the C ABI, and the Python ops when the allocator has no more left."""

from __future__ import annotations

import ctypes

import pytest
import torch

from gpu_util import DEV, TOL, announce, check_grad, check_out, seeded
from kempnerforge_amd import _lib, ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

BF16, F32 = torch.bfloat16, torch.float32
# dtype, B, S, Hq, Hkv, D, a kernel that only a larger workspace runs
CASES = [(BF16, 1, 200, 4, 2, 96, "widen"), (F32, 1, 200, 4, 2, 80, "widen"),
         (F32, 1, 200, 4, 2, 96, "bwd_dkdv_f32"), (F32, 2, 200, 6, 2, 64, "dkdv_parts_f32"),
         (F32, 1, 150, 3, 3, 128, "dkdv_parts_f32")]
IDS = ["-".join(map(str, (str(c[0])[6:],) + c[1:6])) for c in CASES]


def _inputs(dtype, B, S, Hq, Hkv, D):
    q, k, v, do = (seeded((B, S, h, D), i, dtype) for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    return (q, k, v, do) + tuple(ref.rope_tables(D, S, 5e5))


def _check(grads, q, k, v, do, cos, sin):
    want = ref.attention_bwd(q, k, v, cos, sin, do)
    for name, g, w in zip(("dq", "dk", "dv"), grads, want):
        check_grad(g, w, q.dtype, name, group=1 if name == "dq" else q.shape[2] // k.shape[2])


@pytest.mark.parametrize("cfg", CASES, ids=IDS)
def test_backward_with_exactly_the_least(cfg):
    dtype, B, S, Hq, Hkv, D, fast = cfg
    announce(f"least workspace {cfg}")
    q, k, v, do, cos, sin = _inputs(*cfg[:6])
    args = [t.to(DEV) for t in (q, k, v, cos, sin)]
    out, lse = ops.fwd_raw(*args, causal=True, k_rotated=False)
    code, lib = ops._DTYPES[dtype], _lib.load()
    n = _lib.size_out()
    _lib.check(lib.kf_attn_bwd_workspace_size_min(B, S, Hq, Hkv, D, code, ctypes.byref(n)), "size")
    pad = 4096
    ws = torch.full((n.value + pad,), 0xA5, dtype=torch.uint8, device=DEV)
    grads = [torch.empty_like(t) for t in args[:3]]
    p = [t.data_ptr() for t in args + [out, lse, do.to(DEV)] + grads]
    with _lib.KernelTimer() as t:
        _lib.check(lib.kf_attn_bwd(*p, ws.data_ptr(), n.value, B, S, Hq, Hkv, D, 1, None, None,
                                   code, torch.cuda.current_stream().cuda_stream), "kf_attn_bwd")
        torch.cuda.synchronize()
    assert fast not in t.stats, t.stats
    assert (ws[n.value:] == 0xA5).all()
    _check(grads, q, k, v, do, cos, sin)
    rc = lib.kf_attn_bwd(*p, ws.data_ptr(), n.value - 1, B, S, Hq, Hkv, D, 1, None, None, code,
                         torch.cuda.current_stream().cuda_stream)
    assert rc == 4  # KF_ERR_WORKSPACE, before any launch


@pytest.mark.parametrize("cfg", CASES, ids=IDS)
def test_out_of_memory_takes_the_slower_route(cfg, monkeypatch):
    """Allocations above what the least workspace needs fail, as on a full card."""
    dtype, B, S, Hq, Hkv, D, fast = cfg
    announce(f"out of memory {cfg}")
    q, k, v, do, cos, sin = _inputs(*cfg[:6])
    qd, kd, vd = (t.to(DEV).requires_grad_(True) for t in (q, k, v))
    sizes = (0, B, S, Hq, Hkv, D, ops._DTYPES[dtype])
    limit = max(ops._size("kf_attn_bwd_workspace_size_min", *sizes),
                ops._size("kf_attn_fwd_workspace_size_min", *sizes[:2], S, *sizes[2:]))
    empty, refused = torch.empty, []

    def full_card(*a, **kw):
        if kw.get("dtype") is torch.uint8 and a[0] > limit:
            refused.append(a[0])
            raise torch.OutOfMemoryError("no more memory")
        return empty(*a, **kw)

    monkeypatch.setattr(torch, "empty", full_card)
    with _lib.KernelTimer() as t:
        out = ops.attention(qd, kd, vd, cos.to(DEV), sin.to(DEV))
        grads = torch.autograd.grad(out, (qd, kd, vd), do.to(DEV))
        probs = ops.capture_raw(*(x.to(DEV) for x in (q, k, v, cos, sin)), causal=True,
                                k_rotated=False)[1]
        torch.cuda.synchronize()
    monkeypatch.undo()
    assert refused and fast not in t.stats, t.stats
    check_out(out, ref.attention_fwd(q, k, v, cos, sin)[0], TOL[dtype], "out")
    check_out(probs, ref.capture(q, k, v, cos, sin)[1], 1e-5, "probs")
    _check(grads, q, k, v, do, cos, sin)
