"""dQ from the dS records with workgroups of two query tiles and two key slices:
odd numbers of tiles and of record columns, and the sizes on both sides of each
line of the rule that takes them."""

from __future__ import annotations

import pytest
import torch

from gpu_util import DEV, announce, check_grad, kernel_variants, seeded
from kempnerforge_amd import _lib, ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("cfg", [
    # dtype, B, S, Hq, Hkv, D, causal
    (BF16, 1, 193, 3, 3, 128, True),     # four tiles, the last of one row
    (F16, 1, 200, 3, 1, 64, False),      # n_rep 3; seven columns: a slice with none left
    (BF16, 2, 270, 5, 1, 128, True),     # n_rep 5; five tiles: one without a partner
    (BF16, 1, 300, 2, 2, 64, False),
    (BF16, 1, 192, 3, 3, 64, True),      # three tiles: not split
    (BF16, 1, 1000, 2, 1, 64, True),     # two heads, two slices (16 tiles)
    (BF16, 1, 961, 6, 1, 128, False),    # 31 columns
    (BF16, 1, 960, 2, 1, 64, True),      # 15 tiles: not split
    (F16, 2, 2000, 18, 1, 64, True),     # 32 tiles, 576 in all: two tiles and two slices
    (BF16, 5, 2055, 4, 1, 64, True),     # n_rep 4: one tile
    (BF16, 2, 2083, 16, 8, 64, True),    # 33 tiles, one without a partner
    (BF16, 8, 1500, 8, 4, 64, True),     # 384 tiles in rows of 24: not split
    (BF16, 3, 1500, 15, 15, 64, True),   # one head, 540 workgroups of two tiles and slices
    (BF16, 2, 1500, 15, 15, 64, True),   # 360 of them: between one and two per CU, not split
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])))
def test_gradients(cfg):
    dtype, B, S, Hq, Hkv, D, causal = cfg
    announce(f"dq split {cfg}")
    q, k, v, do = (seeded((B, S, h, D), i, dtype) for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    cos, sin = ref.rope_tables(D, S, 5e5)
    args = [t.to(DEV) for t in (q, k, v, cos, sin)]
    out, lse = ops.fwd_raw(*args, causal=causal, k_rotated=False)
    with _lib.KernelTimer() as t:
        dq = ops.bwd_raw(*args, out, lse, do.to(DEV), causal=causal)[0]
        torch.cuda.synchronize()
    assert "bwd_dq_ds" in t.stats, t.stats
    want = ref.attention_bwd(q, k, v, cos, sin, do, causal=causal)[0]
    check_grad(dq, want, dtype, "dq")


@pytest.mark.parametrize("cfg,form", [
    # dtype, B, S, Hq, Hkv, D; heads, query tiles and key slices per workgroup
    ((BF16, 1, 193, 3, 3, 128), (1, 2, 2)),
    ((BF16, 1, 192, 3, 3, 64), (1, 1, 1)),       # three tiles
    ((BF16, 1, 1000, 2, 1, 64), (2, 1, 2)),
    ((BF16, 1, 960, 2, 1, 64), (2, 1, 1)),       # 15 tiles
    ((F16, 2, 2000, 18, 1, 64), (2, 2, 2)),      # 32 tiles, 576 in all
    ((F16, 2, 1980, 18, 1, 64), (2, 1, 1)),      # 31 tiles
    ((BF16, 8, 1500, 8, 4, 64), (2, 1, 1)),
    ((BF16, 4, 1500, 15, 15, 64), (1, 2, 2)),    # 720 workgroups of two tiles and slices
    ((BF16, 3, 1500, 15, 15, 64), (1, 1, 1)),    # 540, but 45 KV heads
    ((BF16, 3, 1500, 12, 12, 64), (1, 1, 1)),    # 432
    ((BF16, 2, 1500, 15, 15, 64), (1, 1, 1)),    # 360
    ((BF16, 5, 2055, 4, 1, 64), (4, 1, 1)),
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])) if len(c) > 3 else
    "x".join(map(str, c)))
@pytest.mark.parametrize("padded", [False, True])
def test_which_form_ran(cfg, form, padded):
    """Key padding takes the unmasked launch's key slices and one tile."""
    dtype, B, S, Hq, Hkv, D = cfg
    announce(f"dq form {cfg} {padded}")
    q, k, v, do = (seeded((B, S, h, D), i, dtype).to(DEV) for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    cos, sin = (t.to(DEV) for t in ref.rope_tables(D, S, 5e5))
    kw = {"key_padding_mask": torch.ones(B, S, dtype=torch.bool, device=DEV)} if padded else {}
    out, lse = ops.fwd_raw(q, k, v, cos, sin, causal=True, k_rotated=False, **kw)
    ran = kernel_variants(lambda: ops.bwd_raw(q, k, v, cos, sin, out, lse, do, causal=True, **kw),
                          "bwd_dq_ds_kernel")
    hb, qt, ksp = form
    # template arguments: D, heads, tiles, slices, mode, ring depth
    assert [r[:4] for r in ran] == [(D, hb, 1 if padded else qt, ksp)], ran
