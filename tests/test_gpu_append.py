"""Prefill append in 16-byte pieces: every type, head sizes of one piece and of
several, batches, offsets, and buffers off 16 bytes (element-wise kernel); the
rows are the oracle's bits and nothing beside them is written."""

from __future__ import annotations

import pytest
import torch

from gpu_util import DEV, announce, seeded
from kempnerforge_amd import ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

BF16, F16, F32 = torch.bfloat16, torch.float16, torch.float32


@pytest.mark.parametrize("cfg", [
    # dtype, B, Snew, Hkv, D, Smax, start, elements the cache is off 16 bytes
    (BF16, 1, 1, 1, 16, 1, 0, 0),       # one thread
    (BF16, 3, 33, 5, 48, 50, 17, 0),    # three pieces per half, last position filled
    (BF16, 2, 40, 3, 40, 64, 3, 0),     # no whole pieces per half
    (BF16, 2, 40, 3, 64, 64, 3, 1),     # unaligned cache
    (F16, 2, 257, 8, 128, 300, 9, 0),
    (F32, 2, 65, 2, 8, 70, 5, 0),
    (F32, 1, 130, 4, 96, 131, 1, 0),
    (F32, 2, 21, 2, 64, 30, 5, 2),
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])))
def test_bits(cfg):
    dtype, B, S, Hkv, D, Smax, start, off = cfg
    announce(f"append {cfg}")
    kn, vn = (seeded((B, S, Hkv, D), i, dtype) for i in (1, 2))
    cos, sin = (t[start:start + S] for t in ref.rope_tables(D, Smax, 5e5))

    def cache():
        n = B * Hkv * Smax * D
        return torch.full((n + 64,), 7.0, dtype=dtype, device=DEV)[off:off + n].view(B, Hkv, Smax, D)

    kc, vc = cache(), cache()
    ops.cache_append_raw(*(t.to(DEV) for t in (kn, vn, cos, sin)), kc, vc, start)
    torch.cuda.synchronize()
    for got, rows in ((kc, ref.apply_rope(kn.transpose(1, 2), cos, sin)), (vc, vn.transpose(1, 2))):
        want = torch.full((B, Hkv, Smax, D), 7.0, dtype=dtype)
        want[:, :, start:start + S] = rows
        assert torch.equal(got.cpu(), want)
