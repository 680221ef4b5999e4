"""The eager shortcut of ``ops.attention`` (an autograd function instead of the
registered operator) against the operator itself, and everything that has to
see the operator: function transforms, forward mode, dispatch modes."""

from __future__ import annotations

import pytest
import torch
from torch.utils._python_dispatch import TorchDispatchMode

from gpu_util import DEV, announce, seeded
from kempnerforge_amd import ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.gpu


def _case(dtype=torch.bfloat16, B=2, S=130, Hq=4, Hkv=2, D=64):
    q, k, v, do = (seeded((B, S, h, D), i, dtype).to(DEV) for i, h in enumerate((Hq, Hkv, Hkv, Hq)))
    cos, sin = (t.to(DEV) for t in ref.rope_tables(D, S, 5e5))
    return [t.requires_grad_(True) for t in (q, k, v)], do, cos, sin


def _op(qkv, cos, sin, **masks):
    return ops.attn_fwd(*qkv, cos, sin, True, masks.get("doc_ids"), masks.get("key_padding_mask"),
                        True)[0]


@pytest.mark.parametrize("dtype,D,mask", [(torch.bfloat16, 64, None), (torch.float16, 128, "doc_ids"),
                                          (torch.bfloat16, 64, "key_padding_mask"),
                                          (torch.float32, 64, None), (torch.bfloat16, 96, None)])
def test_same_bits_as_the_operator(dtype, D, mask):
    announce(f"eager path {dtype} {D} {mask}")
    qkv, do, cos, sin = _case(dtype, D=D)
    masks = {}
    if mask == "doc_ids":
        masks[mask] = (torch.arange(130, device=DEV)[None] // 50).repeat(2, 1)
    elif mask:
        masks[mask] = torch.arange(130, device=DEV)[None] < torch.tensor([[130], [70]], device=DEV)
    a, b = ops.attention(*qkv, cos, sin, **masks), _op(qkv, cos, sin, **masks)
    assert type(a.grad_fn) is not type(b.grad_fn) and torch.equal(a, b)
    for x, y in zip(torch.autograd.grad(a, qkv, do), torch.autograd.grad(b, qkv, do)):
        assert torch.equal(x, y)
    with torch.no_grad():
        c = ops.attention(*qkv, cos, sin, **masks)
    assert not c.requires_grad and torch.equal(c, a)


def test_saved_tensor_hooks_and_no_double_backward():
    announce("eager path hooks")
    qkv, do, cos, sin = _case()
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: (seen.append(t.shape), t.cpu())[1],
                                                  lambda t: t.to(DEV)):
        out = ops.attention(*qkv, cos, sin)
    got = torch.autograd.grad(out, qkv, do)
    assert len(seen) == 6  # rot, v, cos, sin, out, lse
    for x, y in zip(got, torch.autograd.grad(ops.attention(*qkv, cos, sin), qkv, do)):
        assert torch.equal(x, y)
    out = ops.attention(*qkv, cos, sin)
    (dq,) = torch.autograd.grad(out, qkv[:1], do.requires_grad_(True), create_graph=True)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(dq.float().sum(), qkv[1])


def test_modes_and_transforms_get_the_operator():
    announce("eager path modes")
    qkv, do, cos, sin = _case()

    class Seen(TorchDispatchMode):
        names: list = []

        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            self.names.append(str(func))
            return func(*args, **(kwargs or {}))

    with Seen() as m:
        ops.attention(*qkv, cos, sin)
    assert any("kf.attn_fwd" in n for n in m.names)
    # no jvp rule: still refused; vmap still runs the operator per element
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(qkv[0], torch.ones_like(qkv[0]))
        with pytest.raises(Exception):
            ops.attention(dual, *qkv[1:], cos, sin)
    xs = torch.stack([qkv[0], 2 * qkv[0]]).detach()
    kv = [t.detach() for t in qkv[1:]]
    got = torch.func.vmap(lambda x: ops.attention(x, *kv, cos, sin))(xs)
    for x, y in zip(xs, got):
        assert torch.equal(ops.attention(x, *kv, cos, sin), y)
    with pytest.raises(RuntimeError):  # CPU tensors stay refused
        ops.attention(*(t.detach().cpu() for t in qkv), cos, sin)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.float32, 64)])
def test_modes_around_the_backward_get_the_operator(dtype, D):
    announce(f"eager path backward modes {dtype}")
    qkv, do, cos, sin = _case(dtype, D=D)
    dos = torch.stack([do, 2 * do])
    out = ops.attention(*qkv, cos, sin)
    for i in range(2):
        want = torch.autograd.grad(out, qkv, dos[i], retain_graph=True)
        got = torch.autograd.grad(out, qkv, dos, is_grads_batched=True, retain_graph=True)
        for x, y in zip(want, got):
            assert torch.equal(x, y[i])
    names = []

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            names.append(str(func))
            return func(*args, **(kwargs or {}))

    with Seen():
        torch.autograd.grad(out, qkv, do)
    assert any("kf.attn_bwd" in n for n in names)


def test_tables_that_require_a_gradient():
    """Trainable RoPE tables keep the result in the graph, as the operator does,
    with or without trainable q, k and v; they get no gradient."""
    announce("eager path trainable tables")
    qkv, do, cos, sin = _case()
    cos.requires_grad_(True)
    for ts in (qkv, [t.detach() for t in qkv]):
        out = ops.attention(*ts, cos, sin)
        assert out.requires_grad
        out.backward(do)
        assert cos.grad is None
    with torch.no_grad():
        assert not ops.attention(*qkv, cos, sin).requires_grad
