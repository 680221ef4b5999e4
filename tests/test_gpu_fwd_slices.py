"""The forward's two-slice workgroups (small grids): row blocks and key halves
at their edges, halves without a visible key, and the last grid that takes them."""

from __future__ import annotations

import pytest
import torch

from gpu_util import DEV, TOL, announce, check_out, kernel_variants, seeded
from kempnerforge_amd import ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu

BF16, F16 = torch.bfloat16, torch.float16


@pytest.mark.parametrize("cfg", [
    # dtype, B, S, Hq, Hkv, D, causal
    (BF16, 1, 1, 4, 2, 128, True),       # second half empty
    (BF16, 1, 32, 2, 2, 128, True),
    (BF16, 2, 33, 2, 1, 64, False),      # one key in the second half
    (F16, 1, 65, 6, 2, 128, True),       # n_rep 3: 63 of 64 rows; a third half tile
    (BF16, 1, 200, 64, 1, 128, True),    # n_rep 64: one position per block
    (BF16, 1, 200, 80, 1, 64, True),     # n_rep 80: one slice
    (F16, 2, 500, 10, 2, 64, False),
    (BF16, 1, 1024, 32, 8, 128, True),   # 256 blocks (CUs of the chip): two slices
    (BF16, 1, 1028, 32, 8, 128, True),   # one more: one slice
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])))
def test_shapes(cfg):
    dtype, B, S, Hq, Hkv, D, causal = cfg
    announce(f"fwd slices {cfg}")
    q, k, v = (seeded((B, S, h, D), i, dtype) for i, h in enumerate((Hq, Hkv, Hkv)))
    cos, sin = ref.rope_tables(D, S, 5e5)
    args = [t.to(DEV) for t in (q, k, v, cos, sin)]
    out, lse = ops.fwd_raw(*args, causal=causal, k_rotated=False)
    o_ref, l_ref = ref.attention_fwd(q, k, v, cos, sin, causal=causal)
    check_out(out, o_ref, TOL[dtype], "out")
    check_out(lse, l_ref, 1e-3, "lse")
    res = ops.fwd_rot_raw(*args, causal=causal)  # the rotated q rows, stored by both slices
    P = (S + 127) // 128 * 128
    rot_q = res[2][B * Hkv * P * D:].view(B, Hq, P, D)
    assert torch.equal(rot_q[:, :, :S].cpu(), ref.apply_rope(q.transpose(1, 2), cos, sin))
    assert (rot_q[:, :, S:] == 0).all() and torch.equal(res[0], out)


def test_infinite_keys_in_one_half():
    """Scores of -inf over a whole half tile: probability zero there, not NaN,
    whichever half holds them."""
    announce("fwd slices -inf scores")
    B, S, H, D = 1, 64, 1, 64
    cos, sin = torch.ones(S, D // 2), torch.zeros(S, D // 2)  # no rotation
    q = torch.zeros(B, S, H, D, dtype=BF16)
    q[..., 0] = 1.0
    v = seeded((B, S, H, D), 2, BF16)
    for half in (0, 1):
        k = torch.zeros(B, S, H, D, dtype=BF16)
        k[:, 32 * half:32 * half + 32, :, 0] = -float("inf")
        out, _ = ops.fwd_raw(*(t.to(DEV) for t in (q, k, v, cos, sin)), causal=False,
                             k_rotated=True)
        keep = v[:, 32:] if half == 0 else v[:, :32]
        check_out(out, keep.float().mean(1, keepdim=True).expand(B, S, H, D), TOL[BF16], "out")


@pytest.mark.parametrize("cfg,slices", [
    # dtype, B, S, Hq, Hkv, D, causal; r: two-slice workgroups per CU, rounded up
    ((BF16, 1, 63, 4, 2, 128, True), 1),
    ((BF16, 1, 64, 4, 2, 128, True), 2),
    ((BF16, 1, 64, 4, 4, 128, True), 1),      # no groups
    ((BF16, 1, 65, 4, 4, 128, True), 2),
    ((BF16, 1, 200, 64, 1, 128, True), 2),
    ((BF16, 1, 200, 80, 1, 64, True), 1),     # n_rep 80
    ((BF16, 5, 299, 12, 2, 128, True), 1),    # r 2, too short
    ((BF16, 1, 639, 40, 8, 128, True), 1),
    ((BF16, 1, 640, 32, 8, 128, True), 2),
    ((BF16, 1, 1024, 32, 8, 128, False), 2),  # 512 of them
    ((BF16, 1, 1028, 32, 8, 128, True), 1),   # r 3
    ((BF16, 1, 2047, 4, 2, 128, True), 2),
    ((BF16, 1, 2048, 4, 2, 128, True), 1),
    ((BF16, 1, 2048, 4, 2, 64, True), 2),
    ((BF16, 5, 299, 12, 2, 64, True), 1),     # D 64, r 2
    ((BF16, 5, 300, 12, 2, 64, True), 2),
    ((BF16, 4, 599, 16, 16, 64, True), 1),    # r 3
    ((BF16, 4, 600, 16, 16, 64, True), 2),
    ((F16, 4, 1024, 16, 16, 64, True), 1),    # r 4, no groups
    ((F16, 4, 1024, 32, 8, 64, True), 1),     # r 8
    ((F16, 2, 1024, 32, 8, 64, True), 2),     # r 4, groups of four
    ((F16, 2, 1024, 32, 8, 64, False), 1),    # no mask
    ((F16, 5, 1024, 16, 16, 64, True), 2),    # r 5
    ((F16, 6, 1024, 16, 16, 64, True), 1),    # r 6, too short
    ((F16, 3, 2048, 16, 16, 64, True), 2),    # r 6
    ((F16, 2, 3000, 16, 2, 64, True), 1),     # r 6, four groups
    ((F16, 7, 1024, 16, 16, 64, True), 1),    # r 7
], ids=lambda c: "-".join(map(str, (str(c[0])[6:],) + c[1:])) if isinstance(c, tuple) else str(c))
def test_which_form_ran(cfg, slices):
    dtype, B, S, Hq, Hkv, D, causal = cfg
    announce(f"fwd slices form {cfg}")
    q, k, v = (seeded((B, S, h, D), i, dtype).to(DEV) for i, h in enumerate((Hq, Hkv, Hkv)))
    cos, sin = (t.to(DEV) for t in ref.rope_tables(D, S, 5e5))
    ran = kernel_variants(lambda: ops.fwd_raw(q, k, v, cos, sin, causal=causal, k_rotated=False),
                          "fwd32_kernel")
    assert ran == [(D, slices)]


@pytest.mark.parametrize("S,tile", [(64, 0), (64, 1), (128, 0), (128, 1), (128, 3), (300, 2)])
@pytest.mark.parametrize("B", [1, 40])
def test_infinite_keys_in_a_tile(S, tile, B):
    """As above with one slice and with two, wherever the tile of -inf scores is."""
    announce(f"fwd -inf tile {S} {tile} {B}")
    H, D = 8, 64
    cos, sin = torch.ones(S, D // 2), torch.zeros(S, D // 2)  # no rotation
    q = torch.zeros(B, S, H, D, dtype=BF16)
    q[..., 0] = 1.0
    v = seeded((B, S, H, D), 2, BF16)
    k = torch.zeros(B, S, H, D, dtype=BF16)
    gone = slice(32 * tile, 32 * tile + 32)
    k[:, gone, :, 0] = -float("inf")
    args = [t.to(DEV) for t in (q, k, v, cos, sin)]
    out, lse = ops.fwd_raw(*args, causal=False, k_rotated=True)
    kept = torch.ones(S, dtype=torch.bool)
    kept[gone] = False
    want = v[:, kept].float().mean(1, keepdim=True).expand(B, S, H, D)
    check_out(out, want, TOL[BF16], "out")
    check_out(lse, torch.full((B, H, S), float(kept.sum())).log(), 1e-3, "lse")
