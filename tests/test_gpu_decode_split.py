"""The split-K decode's partials over the range of splits per row: from one
chunk in all (fewer chunks than wavefronts, so most of the grid is idle) to
more partials than the merge holds in registers at once."""

from __future__ import annotations

import pytest
import torch

from gpu_util import DEV, announce, max_abs, seeded
from kempnerforge_amd import ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

BF16, F32 = torch.bfloat16, torch.float32


@pytest.mark.parametrize("cfg", [
    # dtype, Hq, Hkv, D, lens: partials per row of the longest sequence
    (BF16, 8, 2, 128, [0]),                  # one chunk per pair
    (BF16, 32, 8, 128, [511]),               # 16: the widest one-wavefront merge
    (BF16, 32, 8, 128, [512]),               # 17: four wavefronts per row
    (BF16, 4, 2, 64, [2048, 31, 32]),        # 65: sixteen, beside one and two
    (BF16, 8, 1, 128, [9000]),               # 282: past the 256 held in registers
    (BF16, 16, 8, 128, [70000]),             # every wavefront of the grid, several chunks each
    (F32, 8, 2, 128, [63]),
    (F32, 8, 2, 64, [1023, 64]),             # 16 splits
    (F32, 8, 2, 128, [1024, 5]),             # 17
    (F32, 4, 1, 128, [19200]),               # 301
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])))
def test_partials(cfg):
    dtype, Hq, Hkv, D, lens = cfg
    announce(f"decode partials {cfg}")
    B, Smax = len(lens), max(lens) + 1
    q = seeded((B, 1, Hq, D), 0, dtype)
    kn = seeded((B, 1, Hkv, D), 1, dtype)
    vn = seeded((B, 1, Hkv, D), 2, dtype)
    kc = seeded((B, Hkv, Smax, D), 5, dtype)
    vc = seeded((B, Hkv, Smax, D), 6, dtype)
    cos, sin = ref.rope_tables(D, Smax, 5e5)
    ln = torch.tensor(lens, dtype=torch.int32)
    kcd, vcd = kc.to(DEV), vc.to(DEV)
    out = ops.decode_raw(q.to(DEV), kn.to(DEV), vn.to(DEV), kcd, vcd, ln.to(DEV), cos.to(DEV),
                         sin.to(DEV), rope_row_offset=0, max_len=Smax)
    torch.cuda.synchronize()
    o_ref, kc_ref, vc_ref = ref.decode_step(q, kn, vn, kc, vc, ln, cos, sin)
    # the output's rounding (bf16: half an ulp of values below 4) and the
    # float32 sums, as for the other decode tests
    assert max_abs(out, o_ref) <= (1e-5 if dtype == F32 else 2e-2)
    assert torch.equal(kcd.cpu(), kc_ref) and torch.equal(vcd.cpu(), vc_ref)
