"""Right-padded batch rows in the 16-bit types, which run the unmasked kernels
with a key limit, and the dealt dK/dV launches: limits at the edges of tiles and
key blocks, blocks wholly past a limit, rows of other layouts beside them."""

from __future__ import annotations

import pytest
import torch

from gpu_util import DEV, TOL, announce, check_grad, check_out, kernel_variants, seeded
from kempnerforge_amd import ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

BF16, F16 = torch.bfloat16, torch.float16
MASK_NONE, MASK_KPM = 0, 2


def _inputs(dtype, B, S, Hq, Hkv, D):
    q, k, v, do = (seeded((B, S, h, D), i, dtype) for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    return (q, k, v, do) + tuple(ref.rope_tables(D, S, 5e5))


def _check(cfg, mask, dkdv):
    """Everything against the oracle, with the dS records and without; ``dkdv``:
    the (LIM, PART, DEAL) of the unmasked dK/dV launch."""
    dtype, B, S, Hq, Hkv, D = cfg
    q, k, v, do, cos, sin = _inputs(*cfg)
    args = [t.to(DEV) for t in (q, k, v, cos, sin)]
    kw = {} if mask is None else {"key_padding_mask": mask}
    kd = {n: m.to(DEV) for n, m in kw.items()}
    out, lse = ops.fwd_raw(*args, causal=True, k_rotated=False, **kd)
    o_ref, l_ref = ref.attention_fwd(q, k, v, cos, sin, **kw)
    check_out(out, o_ref, TOL[dtype], "out")
    check_out(lse, l_ref, 1e-3, "lse")
    want = ref.attention_bwd(q, k, v, cos, sin, do, **kw)
    # short limits leave rows a few keys, where P is near 1 and the rounding of P
    # and dS to the operand type can by itself exceed the base bound (the float64
    # formula with only those roundings: see gpu_util.grad_bound); its error is
    # added to the bound, as in the seeded sweep
    forced = ref.attention_bwd_rounded_operands(q, k, v, cos, sin, do, operand_dtype=dtype, **kw)
    for low in (False, True):
        got = []
        ran = kernel_variants(lambda: got.extend(ops.bwd_raw(
            *args, out, lse, do.to(DEV), causal=True, low_memory=low, **kd)), "bwd_dkdv_kernel")
        # template arguments: D, mode, records kept, LIM, PART, DEAL
        assert [r[3:] for r in ran if r[1] == MASK_NONE] == [dkdv], ran
        assert all(r[0] == D and r[2] == (not low) for r in ran), ran
        for name, g, w, f in zip(("dq", "dk", "dv"), got, want, forced):
            check_grad(g, w, dtype, name, group=1 if name == "dq" else Hq // Hkv, operand_ref=f)
        if mask is not None:  # keys past the limit have no gradient at all
            free = [b for b in range(B) if mask[b, 0]]  # (guarded rows attend padded keys)
            pad = ~mask[free]
            assert (got[1][free].cpu()[pad] == 0).all() and (got[2][free].cpu()[pad] == 0).all()


LIMITS = (1, 33, 300, 63, 64, 65, 299, 127, 128, 129, 32, 255, 256, 257, 31, 192)


@pytest.mark.parametrize("cfg", [
    # dtype, B, S, Hq, Hkv, D: 528 items, unsplit
    (BF16, 22, 300, 16, 8, 128),
    (F16, 22, 300, 8, 8, 64),
    (BF16, 22, 300, 32, 8, 64),
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])))
def test_limits_unsplit(cfg):
    announce(f"right padding {cfg}")
    B, S = cfg[1:3]
    lens = torch.tensor([LIMITS[b % len(LIMITS)] for b in range(B)])
    mask = torch.arange(S)[None, :] < lens[:, None]
    mask[5, 20:30] = False   # a hole: the masked kernels
    mask[6, :7] = False      # guarded rows
    mask[7] = False          # no valid key
    _check(cfg, mask, (1, 0, 1))


@pytest.mark.parametrize("cfg", [
    (BF16, 3, 400, 8, 2, 128),   # small grids: split items
    (F16, 2, 513, 6, 2, 64),
    (BF16, 4, 260, 3, 3, 128),
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])))
@pytest.mark.parametrize("limits", [(1, 129, 128, 200), (64, 257, 31, 1)], ids=str)
def test_limits_split(cfg, limits):
    announce(f"right padding, split {cfg} {limits}")
    B, S = cfg[1:3]
    mask = torch.arange(S)[None, :] < torch.tensor(limits[:B])[:, None]
    _check(cfg, mask, (1, 1, 1))


@pytest.mark.parametrize("cfg,deal", [
    ((BF16, 22, 300, 16, 8, 128), 1),   # three key blocks: dealt
    ((F16, 11, 700, 8, 8, 64), 1),      # six
    ((BF16, 16, 500, 8, 8, 64), 0),     # four, which divide a round: group by group
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])) if isinstance(c, tuple) else str(c))
def test_dealt_without_a_mask(cfg, deal):
    announce(f"dealt dK/dV {cfg}")
    _check(cfg, None, (0, 0, deal))


def test_full_attention_is_not_dealt():
    """Items of equal length: group by group whatever the block count."""
    announce("dealt dK/dV, full attention")
    q, k, v, do, cos, sin = (t.to(DEV) for t in _inputs(BF16, 22, 300, 16, 8, 64))
    out, lse = ops.fwd_raw(q, k, v, cos, sin, causal=False, k_rotated=False)
    ran = kernel_variants(lambda: ops.bwd_raw(q, k, v, cos, sin, out, lse, do, causal=False),
                          "bwd_dkdv_kernel")
    assert [r[1:] for r in ran] == [(MASK_NONE, 1, 0, 0, 0)], ran
