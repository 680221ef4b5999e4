"""Head sizes other than 64 and 128: multiples of 16 up to 128 on the float32
matrix-core kernels (16-bit types and sizes off the multiples of 32 through
float32 copies padded to one), the rest on the generic kernels."""

from __future__ import annotations

import ctypes

import pytest
import torch

from gpu_util import DEV, TOL, announce, check_grad, check_out, max_abs, seeded
from kempnerforge_amd import _lib, ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


def _inputs(dtype, B, S, Hq, Hkv, D):
    q, k, v, do = (seeded((B, S, h, D), i, dtype) for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    return (q, k, v, do) + tuple(ref.rope_tables(D, S, 5e5))


@pytest.mark.parametrize("cfg", [
    # dtype, B, S, Hq, Hkv, D, causal, kernels
    (BF16, 2, 200, 4, 2, 96, True, "wide"),
    (F16, 1, 130, 6, 2, 80, True, "wide"),     # padded 80 -> 96
    (BF16, 1, 257, 8, 1, 112, False, "wide"),  # padded 112 -> 128
    (BF16, 1, 65, 2, 2, 16, True, "wide"),     # padded 16 -> 32: one chunk per half
    (BF16, 2, 33, 4, 4, 48, True, "wide"),
    (F16, 1, 17, 4, 2, 32, True, "wide"),      # the shortest that takes the copies
    (F16, 1, 16, 4, 2, 32, True, "generic"),
    (F16, 1, 1, 4, 2, 32, True, "generic"),    # one token
    (F32, 1, 190, 4, 2, 96, True, "f32"),      # built for float32: no copies
    (F32, 2, 77, 4, 4, 32, False, "f32"),
    (F32, 1, 100, 4, 2, 80, True, "wide"),
    (BF16, 1, 50, 4, 2, 40, True, "generic"),  # no multiple of 16
    (BF16, 1, 50, 2, 1, 160, True, "generic"),  # above 128
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])))
def test_forward_backward(cfg):
    dtype, B, S, Hq, Hkv, D, causal, kernels = cfg
    announce(f"wide {cfg}")
    q, k, v, do, cos, sin = _inputs(dtype, B, S, Hq, Hkv, D)
    args = [t.to(DEV) for t in (q, k, v, cos, sin)]
    with _lib.KernelTimer() as t:
        out, lse = ops.fwd_raw(*args, causal=causal, k_rotated=False)
        res = [ops.bwd_raw(*args, out, lse, do.to(DEV), causal=causal, low_memory=low)
               for low in (False, True)]
        torch.cuda.synchronize()
    ran = set(t.stats)
    assert ("widen" in ran) == (kernels == "wide") and ("fwd_generic" in ran) == (
        kernels == "generic"), ran
    o_ref, l_ref = ref.attention_fwd(q, k, v, cos, sin, causal=causal)
    check_out(out, o_ref, TOL[dtype], "out")
    check_out(lse, l_ref, 1e-5 if dtype == F32 else 1e-3, "lse")
    want = ref.attention_bwd(q, k, v, cos, sin, do, causal=causal)
    for grads in res:  # from the kept dS and recomputing it
        for name, got, w in zip(("dq", "dk", "dv"), grads, want):
            check_grad(got, w, dtype, name, group=1 if name == "dq" else Hq // Hkv)


@pytest.mark.parametrize("mask", ["doc_ids", "key_padding_mask"])
def test_masks(mask):
    B, S, Hq, Hkv, D = 2, 150, 4, 2, 96
    announce(f"wide {mask}")
    q, k, v, do, cos, sin = _inputs(BF16, B, S, Hq, Hkv, D)
    if mask == "doc_ids":
        m = (torch.arange(S)[None, :] // torch.tensor([[47], [64]])).to(torch.int32)
    else:
        m = torch.arange(S)[None, :] >= torch.tensor([[0], [5]])  # row 1: five guarded rows
        m[0, 101:] = False
    qd, kd, vd = (t.to(DEV).requires_grad_(True) for t in (q, k, v))
    out = ops.attention(qd, kd, vd, cos.to(DEV), sin.to(DEV), **{mask: m.to(DEV)})
    grads = torch.autograd.grad(out, (qd, kd, vd), do.to(DEV))
    check_out(out, ref.attention_fwd(q, k, v, cos, sin, causal=True, **{mask: m})[0], TOL[BF16],
              "out")
    want = ref.attention_bwd(q, k, v, cos, sin, do, causal=True, **{mask: m})
    for name, got, w in zip(("dq", "dk", "dv"), grads, want):
        check_grad(got, w, BF16, name, group=1 if name == "dq" else Hq // Hkv)


def test_cache_views_and_capture():
    """Strided rotated keys (a KV cache longer than the queries), and the
    capture's probabilities, whose rows sum to one."""
    B, Sq, Sk, Hq, Hkv, D = 2, 40, 70, 4, 2, 80
    announce("wide cache views")
    q, k, v, _, cos, sin = _inputs(F16, B, Sk, Hq, Hkv, D)
    q = q[:, :Sq].contiguous()
    kc, vc = (t.transpose(1, 2).contiguous().to(DEV) for t in (k, v))  # [B, Hkv, Sk, D]
    out, lse = ops.fwd_raw(q.to(DEV), kc, vc, cos.to(DEV), sin.to(DEV), causal=True,
                           k_rotated=True, k_layout="bhsd")
    o_ref, l_ref = ref.attention_fwd_rotated(q, kc.cpu(), vc.cpu(), cos[:Sq], sin[:Sq])
    check_out(out, o_ref, TOL[F16], "out")
    check_out(lse, l_ref, 1e-3, "lse")
    q2, k2, v2, _, cos, sin = _inputs(F16, B, Sk, Hq, Hkv, D)
    args = [t.to(DEV) for t in (q2, k2, v2, cos, sin)]
    o2, probs, _ = ops.capture_raw(*args, causal=True, k_rotated=False)
    check_out(o2, ref.attention_fwd(q2, k2, v2, cos, sin, causal=True)[0], TOL[F16], "out")
    assert max_abs(probs.sum(-1), torch.ones(B, Hq, Sk)) <= 1e-5
    assert (probs.triu(1) == 0).all()


def test_decode_f32_dims():
    for D in (32, 96):
        announce(f"decode f32 D={D}")
        B, Hq, Hkv, Smax = 2, 8, 2, 400
        lens = torch.tensor([3, 391], dtype=torch.int32)
        q, kn, vn = (seeded((B, 1, h, D), i, F32) for i, h in enumerate((Hq, Hkv, Hkv)))
        kc, vc = (seeded((B, Hkv, Smax, D), i, F32) for i in (5, 6))
        cos, sin = ref.rope_tables(D, Smax, 5e5)
        kcd, vcd = kc.to(DEV), vc.to(DEV)
        out = ops.decode_raw(q.to(DEV), kn.to(DEV), vn.to(DEV), kcd, vcd, lens.to(DEV),
                             cos.to(DEV), sin.to(DEV), rope_row_offset=0, max_len=392)
        o_ref, kc_ref, _ = ref.decode_step(q, kn, vn, kc, vc, lens, cos, sin)
        check_out(out, o_ref, TOL[F32], "out")
        assert torch.equal(kcd.cpu(), kc_ref)


def test_no_workspace():
    """Callers that bring no workspace for these sizes get the generic kernels."""
    announce("wide without a workspace")
    B, S, Hq, Hkv, D = 1, 40, 2, 1, 96
    for dtype, code in ((BF16, _lib.DTYPE_BF16), (F32, _lib.DTYPE_F32)):
        q, k, v, _, cos, sin = _inputs(dtype, B, S, Hq, Hkv, D)
        qd, kd, vd, cd, sd = (t.to(DEV) for t in (q, k, v, cos, sin))
        out = torch.empty_like(qd)
        p = lambda t: ctypes.c_void_p(t.data_ptr())  # noqa: E731
        st = (S * Hkv * D, Hkv * D, D)
        _lib.check(_lib.load().kf_attn_fwd(
            p(qd), p(kd), p(vd), p(cd), p(sd), p(out), None, None, 0, B, S, S, Hq, Hkv, D, *st,
            *st, 0, 1, None, None, code,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), "kf_attn_fwd")
        torch.cuda.synchronize()
        check_out(out, ref.attention_fwd(q, k, v, cos, sin, causal=True)[0], TOL[dtype], "out")
