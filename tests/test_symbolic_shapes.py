"""Tracing ``ops.attention`` with symbolic sizes.  The fake kernels run on the
CPU, so this needs the built library (kf_attn_rot_size) and no GPU."""

from __future__ import annotations

import os

import pytest
import torch
from torch.fx.experimental.proxy_tensor import make_fx

from kempnerforge_amd import _lib, ops
from oracle import attention_ref as ref

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="library not built")


def _train(q, k, v, cos, sin, do):
    out = ops.attention(q, k, v, cos, sin)
    return (out,) + torch.autograd.grad(out, (q, k, v), do)


@pytest.mark.parametrize("dtype,D", [(torch.bfloat16, 64), (torch.float32, 64),
                                     (torch.bfloat16, 96)])
def test_symbolic_trace_of_a_training_step(dtype, D):
    """Sizes reach the fake kernels as SymInts, and rot_size among them."""
    for S in (250, 300):
        q, k, v, do = (torch.randn(2, S, h, D, dtype=dtype) for h in (4, 2, 2, 4))
        qkv = [t.requires_grad_(True) for t in (q, k, v)]
        g = make_fx(_train, tracing_mode="symbolic")(*qkv, *ref.rope_tables(D, S, 5e5), do)
        targets = [str(n.target) for n in g.graph.nodes if n.op == "call_function"]
        assert "kf.attn_fwd.default" in targets
        assert ("kf.attn_bwd_rot.default" if ops.rot_size(2, S, 4, 2, D, dtype, False, False)
                else "kf.attn_bwd.default") in targets


@pytest.mark.gpu
@pytest.mark.parametrize("dynamic", [None, True])
def test_compiled_training_at_several_lengths(dynamic):
    """A second length makes torch.compile's sizes symbolic by itself."""
    from gpu_util import DEV, announce, seeded

    announce(f"compile, dynamic={dynamic}")
    torch._dynamo.reset()
    f = torch.compile(lambda q, k, v, c, s: ops.attention(q, k, v, c, s).float().square().sum(),
                      fullgraph=True, backend="aot_eager", dynamic=dynamic)
    for S in (250, 300, 333):
        q, k, v = (seeded((1, S, h, 64), h, torch.bfloat16).to(DEV).requires_grad_(True)
                   for h in (4, 2, 2))
        cos, sin = (t.to(DEV) for t in ref.rope_tables(64, S, 5e5))
        got = torch.autograd.grad(f(q, k, v, cos, sin), (q, k, v))
        want = torch.autograd.grad(ops.attention(q, k, v, cos, sin).float().square().sum(),
                                   (q, k, v))
        for a, b in zip(got, want):
            assert torch.equal(a, b)
