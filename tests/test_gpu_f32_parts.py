"""The float32 dK/dV pass split into heads and runs of query tiles (small grids)
beside the unsplit one: runs of unequal and of no tiles, every mask, and the
sizes on both sides of the split."""

from __future__ import annotations

import pytest
import torch

from gpu_util import DEV, announce, check_grad, seeded
from kempnerforge_amd import _lib, ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

F32 = torch.float32


@pytest.mark.parametrize("cfg", [
    # B, S, Hq, Hkv, D, causal, mask, split
    (1, 33, 2, 2, 64, True, None, True),     # two tiles, two runs
    (1, 500, 6, 2, 128, True, None, True),   # 16 tiles over 8 runs; late key blocks have fewer tiles
    (2, 190, 4, 1, 32, False, None, True),
    (1, 300, 8, 2, 64, True, "doc", True),   # listed tiles: runs of one or none
    (2, 200, 4, 2, 96, True, "kpm", True),   # guarded rows' tiles
    (16, 130, 16, 16, 64, True, None, False),  # 768 items, no groups
    (16, 130, 32, 16, 64, True, None, True),   # the same items in groups of two: heads only
    (22, 130, 16, 16, 64, True, "doc", False),  # 1056 items
    # without groups: a line in the positions by items per CU
    (1, 65, 32, 32, 64, True, None, True),      # 64 items
    (1, 90, 40, 40, 64, True, None, False),     # 80: 96 positions
    (1, 96, 40, 40, 64, True, None, True),
    (1, 250, 40, 40, 32, True, None, False),    # 160: 256
    (1, 256, 40, 40, 32, True, None, True),
    (1, 256, 40, 40, 32, False, None, False),   # full attention: 640
    (1, 640, 16, 16, 32, False, None, True),
    (2, 250, 40, 40, 32, True, None, False),    # 320: 256
    (2, 256, 40, 40, 32, True, None, True),
    (2, 600, 20, 20, 32, True, None, False),    # 400: 640
    (2, 640, 20, 20, 32, True, None, True),
    (2, 640, 16, 16, 32, False, None, False),
    (1, 600, 12, 12, 32, True, "doc", False),   # 120: 640
    (1, 640, 12, 12, 32, True, "doc", True),
    (1, 640, 16, 16, 32, True, "doc", False),   # 160
    (2, 640, 16, 16, 32, True, "kpm", True),    # key padding as without a mask
], ids=lambda c: "-".join(map(str, c)))
def test_gradients(cfg):
    B, S, Hq, Hkv, D, causal, mask, split = cfg
    announce(f"f32 parts {cfg}")
    q, k, v, do = (seeded((B, S, h, D), i, F32) for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    cos, sin = ref.rope_tables(D, S, 5e5)
    masks = {}
    if mask == "doc":
        masks["doc_ids"] = ((torch.arange(S)[None, :] + 13 * torch.arange(B)[:, None]) // 45).int()
    elif mask == "kpm":
        m = torch.arange(S)[None, :] >= 40 * torch.arange(B)[:, None]  # row 1: 40 guarded rows
        m[:, 150:] = False
        masks["key_padding_mask"] = m
    args = [t.to(DEV) for t in (q, k, v, cos, sin)]
    md = {n: t.to(DEV) for n, t in masks.items()}
    out, lse = ops.fwd_raw(*args, causal=causal, k_rotated=False, **md)
    with _lib.KernelTimer() as t:
        grads = [ops.bwd_raw(*args, out, lse, do.to(DEV), causal=causal, low_memory=low, **md)
                 for low in (False, True)]
        torch.cuda.synchronize()
    assert ("dkdv_parts_f32" in t.stats) == split, t.stats
    want = ref.attention_bwd(q, k, v, cos, sin, do, causal=causal, **masks)
    for got in grads:
        for name, g, w in zip(("dq", "dk", "dv"), got, want):
            check_grad(g, w, F32, name, group=1 if name == "dq" else Hq // Hkv)
    assert torch.equal(grads[0][1], grads[1][1]) and torch.equal(grads[0][2], grads[1][2])
