"""Captures small enough that the probabilities are formed after the forward,
one workgroup per piece of P, beside ones of the fused kernel: row lengths off
the 16-byte alignment and off the 64-key tiles, keys past the last query, one
query over a cache."""

from __future__ import annotations

import pytest
import torch

from gpu_util import DEV, announce, kernel_variants, max_abs, seeded
from kempnerforge_amd import _lib, ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("cfg", [
    # dtype, B, S, Hq, Hkv, D, causal, kernel
    (BF16, 1, 1, 4, 2, 128, True, "after"),
    (BF16, 1, 63, 4, 4, 64, True, "after"),
    (BF16, 1, 65, 8, 2, 128, False, "after"),   # one key in the last tile
    (F16, 2, 257, 6, 2, 128, True, "after"),    # a second chunk of one key; n_rep 3
    (BF16, 1, 516, 5, 1, 64, True, "after"),    # rows 16-byte aligned, n_rep 5
    (BF16, 1, 770, 4, 1, 128, True, "after"),   # zero-only chunks; odd row starts
    (BF16, 16, 67, 16, 16, 64, True, "fused"),   # fused, unaligned rows
    (F16, 32, 130, 16, 8, 128, False, "fused"),
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])))
def test_shapes(cfg):
    dtype, B, S, Hq, Hkv, D, causal, kernel = cfg
    announce(f"small capture {cfg}")
    q, k, v = (seeded((B, S, h, D), i, dtype) for i, h in enumerate((Hq, Hkv, Hkv)))
    cos, sin = ref.rope_tables(D, S, 5e5)
    args = [t.to(DEV) for t in (q, k, v, cos, sin)]
    with _lib.KernelTimer() as t:
        out, p, lse = ops.capture_raw(*args, causal=causal, k_rotated=False)
        torch.cuda.synchronize()
    assert ("fwd_mfma" in t.stats) == (kernel == "after"), t.stats
    o_ref, p_ref = ref.capture(q, k, v, cos, sin, causal=causal)
    assert max_abs(p, p_ref) <= 1e-5
    if causal:
        assert (p.triu(1) == 0).all()
    assert max_abs(out, o_ref) <= (2e-2 if dtype == BF16 else 5e-3)
    assert max_abs(lse, ref.attention_fwd(q, k, v, cos, sin, causal=causal)[1]) <= 1e-3


@pytest.mark.parametrize("Sq,causal", [(1, False), (30, True)])
def test_cache(Sq, causal):
    """Rotated keys in a cache view longer than the queries (top-left causal)."""
    announce(f"small capture over a cache, {Sq} queries")
    B, Sk, Hq, Hkv, D = 2, 203, 8, 2, 128
    q = seeded((B, Sq, Hq, D), 0, BF16)
    kc, vc = (seeded((B, Hkv, Sk + 5, D), i, BF16) for i in (1, 2))
    cos, sin = ref.rope_tables(D, Sq, 5e5)
    kd, vd = (t.to(DEV)[:, :, :Sk] for t in (kc, vc))
    out, p, _ = ops.capture_raw(q.to(DEV), kd, vd, cos.to(DEV), sin.to(DEV), causal=causal,
                                k_rotated=True, k_layout="bhsd")
    o_ref, l_ref = ref.attention_fwd_rotated(q, kc[:, :, :Sk], vc[:, :, :Sk], cos, sin,
                                             causal=causal)
    assert max_abs(out, o_ref) <= 2e-2
    qr = ref.apply_rope(q.transpose(1, 2), cos, sin).double()
    s = qr @ kc[:, :, :Sk].double().repeat_interleave(Hq // Hkv, 1).transpose(2, 3) * D ** -0.5
    if causal:
        s = s.masked_fill(torch.ones(Sq, Sk, dtype=torch.bool).triu(1), float("-inf"))
    assert max_abs(p, torch.softmax(s, -1)) <= 1e-5


P_NT, P_VEC, P_ANY = 0, 1, 2  # non-temporal, 16-byte write-back, and stores with a tail


@pytest.mark.parametrize("S,pst", [(144, P_NT), (148, P_VEC), (150, P_ANY), (151, P_ANY)])
@pytest.mark.parametrize("mask", [None, "doc_ids", "key_padding_mask"])
@pytest.mark.parametrize("D", [64, 128])
def test_stores_of_the_fused_kernel(S, pst, mask, D):
    announce(f"fused capture stores S={S} {mask} D={D}")
    B, Hq, Hkv = (30, 16, 16) if mask is None else (2, 6, 2)
    q, k, v = (seeded((B, S, h, D), i, BF16) for i, h in enumerate((Hq, Hkv, Hkv)))
    cos, sin = ref.rope_tables(D, S, 5e5)
    m = {}
    if mask == "doc_ids":
        m[mask] = (torch.arange(S)[None, :] // torch.tensor([[47], [64]])).to(torch.int32)
    elif mask:
        m[mask] = torch.arange(S)[None, :] >= torch.tensor([[0], [9]])  # row 1: guarded rows
        m[mask][0, 70:] = False
    args = [t.to(DEV) for t in (q, k, v, cos, sin)]
    got = []
    ran = kernel_variants(lambda: got.extend(ops.capture_raw(
        *args, causal=True, k_rotated=False, **{n: t.to(DEV) for n, t in m.items()})),
        "capture_probs_mfma_kernel")
    assert [(r[0], r[2]) for r in ran] == [(D, pst)], ran
    o_ref, p_ref = ref.capture(q, k, v, cos, sin, **m)
    assert max_abs(got[1], p_ref) <= 1e-5 and max_abs(got[0], o_ref) <= 2e-2
    assert got[1].cpu()[p_ref == 0].abs().max().item() == 0.0


@pytest.mark.parametrize("cfg,after", [
    ((1, 1200, 32, 8, 64), True),    # 176 MiB of P
    ((1, 1300, 32, 8, 64), False),   # 206, rows off 64-byte blocks
    ((1, 1600, 32, 8, 64), True),    # 312, whole blocks
    ((1, 1632, 32, 8, 64), False),   # 325
    ((2, 1000, 32, 8, 64), False),   # 256 workgroups of the fused kernel
], ids=lambda c: "-".join(map(str, c)) if isinstance(c, tuple) else str(c))
def test_which_form_ran(cfg, after):
    B, S, Hq, Hkv, D = cfg
    announce(f"capture form {cfg}")
    q, k, v = (seeded((B, S, h, D), i, BF16).to(DEV) for i, h in enumerate((Hq, Hkv, Hkv)))
    cos, sin = (t.to(DEV) for t in ref.rope_tables(D, S, 5e5))
    got = []
    ran = kernel_variants(lambda: got.extend(ops.capture_raw(q, k, v, cos, sin, causal=True,
                                                             k_rotated=False)),
                          "capture_tiles_kernel")
    assert len(ran) == after
    assert max_abs(got[1].sum(-1), torch.ones(B, Hq, S)) <= 1e-5 and (got[1].triu(1) == 0).all()
