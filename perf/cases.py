"""The attention calls whose speed this repository answers for, on one GPU.

Each case is one attention layer's work in training, prefill, decode or
capture, through the calls a user's program makes (``ops.attention`` under
autograd, ``ops.cache_append_raw`` + ``ops.fwd_raw``, ``ops.decode_raw``,
``ops.capture_raw`` and the ``Attention`` module), from the smallest
configuration the repository names to the largest.  ``listed`` gives the fixed
cases, ``draw`` more of the same ranges; ``prepare`` makes a case's inputs on
the GPU, ``run`` is one pass, ``exact`` the same results in 64 bits from plain
torch, ``work`` the bytes and operations a pass cannot do without.
"""

import math

import torch

from kempnerforge_amd import Attention, ops
from kempnerforge_amd.position import precompute_rope_frequencies

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
THETA = 500000.0


def _train(name, B, S, Hq, Hkv, D, dtype="bf16", mask="none"):
    return {"name": name, "kind": "train", "B": B, "S": S, "Hq": Hq, "Hkv": Hkv, "D": D,
            "dtype": dtype, "mask": mask}


def listed():
    return [
        # The debug configuration's layer (256-token context, two KV heads) in
        # float32: what a user steps through first, launches and latency only.
        _train("train_debug_fp32", 2, 256, 4, 2, 64, "fp32"),
        # Forward and backward of an 8B layer, the training configuration of
        # the repository's benchmark.
        _train("train_8b", 4, 4096, 32, 8, 128),
        # The same layer on packed documents, how pre-training batches are made.
        _train("train_8b_docs", 4, 4096, 32, 8, 128, mask="docs"),
        # A multimodal batch of samples of unequal length, padded on the right,
        # in float16; an odd sequence length, as the longest sample gives it.
        _train("train_padded_fp16", 6, 1531, 32, 8, 128, "fp16", mask="padding"),
        # One rank's share of a 13B layer under 4-way tensor parallelism: few
        # heads, and five query heads per KV head (no power of two).
        _train("train_tp4_share", 2, 4096, 10, 2, 128),
        # Long-context training, the 70B layer at 16384 tokens: the largest.
        _train("train_70b_long", 1, 16384, 64, 8, 128),
        # A model whose dim / n_heads is neither 64 nor 128 (here 96).
        _train("train_d96", 2, 1024, 16, 16, 96),
        # The reference's attention micro-benchmark: the whole module
        # (projections included) of a 768-wide model, inference.
        {"name": "module_768", "kind": "module", "B": 4, "S": 512, "Hq": 12, "Hkv": 12, "D": 64,
         "dtype": "bf16"},
        # Prefill of one prompt of odd length into a fresh KV cache, 8B layer.
        {"name": "prefill_prompt", "kind": "prefill", "B": 1, "S": 1999, "Hq": 32, "Hkv": 8,
         "D": 128, "dtype": "bf16"},
        # The next token of one interactive generation: the smallest call.
        {"name": "decode_single", "kind": "decode", "B": 1, "L": 1000, "Hq": 32, "Hkv": 8,
         "D": 128, "dtype": "bf16", "qk_norm": False},
        # A serving batch of 32 sequences of 1024 to 8192 tokens.
        {"name": "decode_batch", "kind": "decode", "B": 32, "L": 8192, "Hq": 32, "Hkv": 8,
         "D": 128, "dtype": "bf16", "qk_norm": False},
        # Attention probabilities of one short text, as a notebook looks at
        # them: odd length, so that the rows of P are not aligned.
        {"name": "capture_text", "kind": "capture", "B": 1, "S": 777, "Hq": 32, "Hkv": 8,
         "D": 128, "dtype": "bf16"},
    ]


# (Hq, Hkv, D) of the configurations the repository names: the 8B and 70B
# layers, shares of 4-way tensor parallelism, the micro-benchmark, small models
HEADS = [(32, 8, 128), (64, 8, 128), (16, 2, 128), (12, 2, 128), (10, 2, 128), (8, 2, 128),
         (12, 12, 64), (4, 2, 64), (16, 16, 64), (32, 8, 64)]
HEADS_OTHER_D = [(16, 16, 96), (8, 2, 32), (12, 4, 80)]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["train", "train", "train", "module", "prefill", "decode", "decode",
                       "capture"])
    Hq, Hkv, D = rng.choice(HEADS)
    dtype = rng.choice(["bf16", "bf16", "bf16", "bf16", "fp16", "fp32"])
    if kind == "train":
        mask = rng.choice(["none", "none", "docs", "padding"])
        if rng.random() < 0.15:
            (Hq, Hkv, D), mask = rng.choice(HEADS_OTHER_D), "none"
            dtype = rng.choice(["bf16", "fp16"])
        small = dtype == "fp32" or D not in (64, 128)
        S = _log_int(rng, 65, 1024 if small else 4096)
        B = rng.randint(1, max(1, min(8, (2048 if small else 16384) // S)))
        return {"kind": kind, "B": B, "S": S, "Hq": Hq, "Hkv": Hkv, "D": D, "dtype": dtype,
                "mask": mask}
    if kind == "decode":
        B = _log_int(rng, 1, 64)
        return {"kind": kind, "B": B, "L": _log_int(rng, 33, min(32768, 262144 // B)), "Hq": Hq,
                "Hkv": Hkv, "D": D, "dtype": dtype, "qk_norm": rng.random() < 0.3}
    if kind == "module":
        S = _log_int(rng, 33, 2048)
        return {"kind": kind, "B": rng.randint(1, max(1, min(8, 4096 // S))), "S": S, "Hq": Hq,
                "Hkv": Hkv, "D": D, "dtype": "bf16" if dtype == "fp32" else dtype}
    if kind == "prefill":
        S = _log_int(rng, 17, 2048 if dtype == "fp32" else 8192)
        B = rng.randint(1, max(1, min(8, 8192 // S)))
        return {"kind": kind, "B": B, "S": S, "Hq": Hq, "Hkv": Hkv, "D": D, "dtype": dtype}
    return {"kind": kind, "B": 1, "S": _log_int(rng, 50, 2048), "Hq": Hq, "Hkv": Hkv, "D": D,
            "dtype": dtype}


# ------------------------------------------------------------------ layouts
def _doc_lengths(case, seed):
    """Per batch row, the lengths of the documents packed into it (log-uniform
    from 32 tokens to the context)."""
    g = torch.Generator().manual_seed(1000003 * seed + case["S"])
    S, rows = case["S"], []
    for _ in range(case["B"]):
        row, left = [], S
        while left > 0:
            u = float(torch.rand((), generator=g))
            n = min(left, int(round(math.exp(math.log(32) + u * math.log(max(S, 64) / 32)))))
            row.append(n)
            left -= n
        rows.append(row)
    return rows


def _valid_lengths(case, seed):
    """Per batch row, the tokens before the padding: the longest sample fills
    the row, the others from a third of it on."""
    g = torch.Generator().manual_seed(1000003 * seed + case["S"])
    S, B = case["S"], case["B"]
    lens = [S - int(float(torch.rand((), generator=g)) * (2 * S // 3)) for _ in range(B)]
    lens[int(float(torch.rand((), generator=g)) * B) % B] = S
    return lens


def _cache_lengths(case, seed):
    """Tokens already cached per sequence (the new one makes at most L)."""
    B, L = case["B"], case["L"]
    if B == 1:
        return [L - 1]
    g = torch.Generator().manual_seed(1000003 * seed + L)
    lo = max(1, L // 8)
    lens = [lo + int(float(torch.rand((), generator=g)) * (L - lo)) for _ in range(B)]
    lens[0] = L - 1
    return lens


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    dt, kind = DTYPES[case["dtype"]], case["kind"]
    B, Hq, Hkv, D = case["B"], case["Hq"], case["Hkv"], case["D"]

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32).to(dt)

    if kind == "decode":
        L = case["L"]
        cos, sin = precompute_rope_frequencies(D, L, THETA, device=torch.device(DEV))
        st = {"kind": kind, "q": rand(B, 1, Hq, D), "k": rand(B, 1, Hkv, D),
              "v": rand(B, 1, Hkv, D), "k_cache": rand(B, Hkv, L, D),
              "v_cache": rand(B, Hkv, L, D), "cos": cos, "sin": sin, "max_len": L,
              "lens": torch.tensor(_cache_lengths(case, seed), dtype=torch.int32, device=DEV),
              "q_norm": None, "k_norm": None}
        if case["qk_norm"]:
            st["q_norm"] = 1 + 0.1 * rand(D).float()
            st["k_norm"] = 1 + 0.1 * rand(D).float()
        return st
    S = case["S"]
    cos, sin = precompute_rope_frequencies(D, S, THETA, device=torch.device(DEV))
    if kind == "module":
        with torch.device("meta"):
            layer = Attention(Hq * D, Hq, Hkv, D)
        layer = layer.to_empty(device=DEV).to(dt).requires_grad_(False).eval()
        for p in layer.parameters():
            p.copy_(rand(*p.shape) * (Hq * D) ** -0.5)
        return {"kind": kind, "layer": layer, "x": rand(B, S, Hq * D), "cos": cos, "sin": sin}
    st = {"kind": kind, "q": rand(B, S, Hq, D), "k": rand(B, S, Hkv, D),
          "v": rand(B, S, Hkv, D), "cos": cos, "sin": sin}
    if kind == "prefill":
        st["k_cache"] = torch.zeros(B, Hkv, S + 256, D, dtype=dt, device=DEV)
        st["v_cache"] = torch.zeros(B, Hkv, S + 256, D, dtype=dt, device=DEV)
    if kind == "train":
        st["dout"] = rand(B, S, Hq, D)
        for name in ("q", "k", "v"):
            st[name].requires_grad_(True)
        st["docs"] = st["valid"] = None
        if case["mask"] == "docs":
            ids = [torch.repeat_interleave(torch.arange(len(row)), torch.tensor(row))
                   for row in _doc_lengths(case, seed)]
            st["docs"] = torch.stack(ids).to(torch.int32).to(DEV)
        elif case["mask"] == "padding":
            lens = torch.tensor(_valid_lengths(case, seed))
            st["valid"] = (torch.arange(S)[None, :] < lens[:, None]).to(DEV)
    return st


def run(state):
    st = state
    if st["kind"] == "train":
        out = ops.attention(st["q"], st["k"], st["v"], st["cos"], st["sin"], causal=True,
                            doc_ids=st["docs"], key_padding_mask=st["valid"])
        dq, dk, dv = torch.autograd.grad(out, (st["q"], st["k"], st["v"]), st["dout"])
        return {"out": out, "dq": dq, "dk": dk, "dv": dv}
    if st["kind"] == "module":
        with torch.no_grad():
            return {"out": st["layer"](st["x"], st["cos"], st["sin"])}
    if st["kind"] == "prefill":
        S, kc, vc = st["q"].shape[1], st["k_cache"], st["v_cache"]
        ops.cache_append_raw(st["k"], st["v"], st["cos"], st["sin"], kc, vc, 0)
        out, _ = ops.fwd_raw(st["q"], kc[:, :, :S], vc[:, :, :S], st["cos"], st["sin"],
                             causal=True, k_rotated=True, k_layout="bhsd")
        return {"out": out, "k_cache": kc, "v_cache": vc}
    if st["kind"] == "decode":
        out = ops.decode_raw(st["q"], st["k"], st["v"], st["k_cache"], st["v_cache"], st["lens"],
                             st["cos"], st["sin"], rope_row_offset=0, max_len=st["max_len"],
                             q_norm_weight=st["q_norm"], k_norm_weight=st["k_norm"])
        return {"out": out, "k_cache": st["k_cache"], "v_cache": st["v_cache"]}
    out, probs, lse = ops.capture_raw(st["q"], st["k"], st["v"], st["cos"], st["sin"],
                                      causal=True, k_rotated=False)
    return {"out": out, "probs": probs, "lse": lse}


# ------------------------------------------------------------------ work and tolerance
def _visible_pairs(case):
    """(query, key) pairs that attention over the whole batch row computes, per
    query head, summed over the batch (masked cases: for the layout of seed 0)."""
    B, S = case["B"], case["S"]
    if case.get("mask") == "docs":
        return sum(n * (n + 1) // 2 for row in _doc_lengths(case, 0) for n in row)
    if case.get("mask") == "padding":
        return sum(n * (n + 1) // 2 + (S - n) * n for n in _valid_lengths(case, 0))
    return B * S * (S + 1) // 2


def work(case):
    B, Hq, Hkv, D = case["B"], case["Hq"], case["Hkv"], case["D"]
    el = 4 if case["dtype"] == "fp32" else 2
    if case["kind"] == "decode":
        keys = sum(n + 1 for n in _cache_lengths(case, 0))
        return {"bytes": el * (2 * keys * Hkv * D + 2 * B * Hq * D + 2 * B * Hkv * D),
                "flops": 4 * D * Hq * keys}
    S = case["S"]
    q, kv = el * B * S * Hq * D, el * B * S * Hkv * D
    fwd = 4 * D * Hq * _visible_pairs(case)
    if case["kind"] == "train":
        # in: q, k, v, dout; out: out, dq, dk, dv.  Backward: S, dP, dV, dK, dQ.
        return {"bytes": 4 * q + 4 * kv, "flops": fwd * 14 // 4}
    if case["kind"] == "module":
        # in: x and the four weights; out: the layer's output
        wts = el * (2 * Hq + 2 * Hkv) * D * Hq * D
        return {"bytes": 2 * q + wts, "flops": fwd + 2 * B * S * wts // el}
    if case["kind"] == "prefill":
        return {"bytes": 2 * q + 4 * kv, "flops": fwd}  # in: q, k, v; out: out and the cache rows
    return {"bytes": 2 * q + 2 * kv + 4 * B * Hq * S * (S + 1), "flops": fwd}


def tolerance(case):
    # About four times what two correct orders of the same sums differ by (the
    # backward from kept dS tiles against the recomputing one, split against
    # unsplit decode): the rounding of P, dS and the results to the storage type.
    if case["dtype"] == "bf16":
        return {"rel": 1e-2}
    if case["dtype"] == "fp16":
        return {"rel": 2e-3}
    return {"rel": 1e-5}


# ------------------------------------------------------------------ 64 bits
def _rotate(x, cos, sin):
    """RoPE of ``x [..., S, H, D]`` in 64 bits, half-split pairs."""
    half = x.shape[-1] // 2
    c, s = cos.double()[:, None, :], sin.double()[:, None, :]
    x1, x2 = x[..., :half], x[..., half:]
    return torch.cat([x1 * c - x2 * s, x2 * c + x1 * s], dim=-1)


def _visible(case, seed, b):
    """Boolean ``[S, S]``: may query i of batch row b attend key j?"""
    S = case["S"]
    pos = torch.arange(S, device=DEV)
    see = pos[:, None] >= pos[None, :]
    if case.get("mask") == "docs":
        row = _doc_lengths(case, seed)[b]
        ids = torch.repeat_interleave(torch.arange(len(row)), torch.tensor(row)).to(DEV)
        see &= ids[:, None] == ids[None, :]
    elif case.get("mask") == "padding":
        see &= (pos < _valid_lengths(case, seed)[b])[None, :]
    return see


def _attend(case, seed, q, k, v, dout=None, keep=False):
    """Attention of rotated ``q, k`` and ``v`` ``[B, S, H, D]`` in 64 bits, one
    query head at a time; with ``dout`` also the gradients of q, k (rotated)
    and v; with ``keep`` also the probabilities and log-sum-exps."""
    B, S, Hq, D = q.shape
    rep = Hq // k.shape[2]
    out = torch.empty_like(q)
    dq, dk, dv = (None, None, None) if dout is None else (
        torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v))
    probs = torch.empty(B, Hq, S, S, dtype=torch.float64, device=DEV) if keep else None
    lse = torch.empty(B, Hq, S, dtype=torch.float64, device=DEV) if keep else None
    for b in range(B):
        hidden = ~_visible(case, seed, b)
        for h in range(Hq):
            qh, kh, vh = q[b, :, h], k[b, :, h // rep], v[b, :, h // rep]
            s = (qh @ kh.T).mul_(D ** -0.5).masked_fill_(hidden, -math.inf)
            if keep:
                lse[b, h] = torch.logsumexp(s, dim=-1)
            p = torch.softmax(s, dim=-1)
            del s
            out[b, :, h] = p @ vh
            if keep:
                probs[b, h] = p
            if dout is not None:
                do = dout[b, :, h]
                dv[b, :, h // rep] += p.T @ do
                ds = do @ vh.T
                ds -= (do * out[b, :, h]).sum(-1, keepdim=True)
                ds *= p
                ds *= D ** -0.5
                dq[b, :, h] = ds @ kh
                dk[b, :, h // rep] += ds.T @ qh
                del ds
            del p
    return out, dq, dk, dv, probs, lse


def _normed(x, w, eps=1e-5):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def exact(case, seed):
    st = prepare(case, seed)
    with torch.no_grad():
        cos, sin, kind = st["cos"], st["sin"], case["kind"]
        if kind == "decode":
            q, k = st["q"].double(), st["k"].double()
            if case["qk_norm"]:
                q, k = _normed(q, st["q_norm"]), _normed(k, st["k_norm"])
            kc, vc = st["k_cache"].double(), st["v_cache"].double()
            out = torch.empty_like(q)
            rep = case["Hq"] // case["Hkv"]
            for b, n in enumerate(_cache_lengths(case, seed)):
                kc[b, :, n] = _rotate(k[b], cos[n:n + 1], sin[n:n + 1])[0]
                vc[b, :, n] = st["v"][b, 0].double()
                qb = _rotate(q[b], cos[n:n + 1], sin[n:n + 1])[0].view(-1, rep, case["D"])
                p = torch.softmax(qb @ kc[b, :, :n + 1].transpose(1, 2) * case["D"] ** -0.5, -1)
                out[b, 0] = (p @ vc[b, :, :n + 1]).reshape(-1, case["D"])
            return {"out": out, "k_cache": kc, "v_cache": vc}
        if kind == "module":
            x, layer = st["x"].double(), st["layer"]
            B, S, _ = x.shape
            q, k, v = ((x @ m.weight.double().T).view(B, S, -1, case["D"])
                       for m in (layer.q_proj, layer.k_proj, layer.v_proj))
            out = _attend(case, seed, _rotate(q, cos, sin), _rotate(k, cos, sin), v)[0]
            return {"out": out.reshape(B, S, -1) @ layer.o_proj.weight.double().T}
        q, k = _rotate(st["q"].double(), cos, sin), _rotate(st["k"].double(), cos, sin)
        v = st["v"].double()
        if kind == "train":
            out, dq, dk, dv, _, _ = _attend(case, seed, q, k, v, st["dout"].double())
            # the rotation's adjoint turns the gradients back
            return {"out": out, "dq": _rotate(dq, cos, -sin), "dk": _rotate(dk, cos, -sin),
                    "dv": dv}
        if kind == "prefill":
            kc, vc = st["k_cache"].double(), st["v_cache"].double()
            kc[:, :, :case["S"]] = k.transpose(1, 2)
            vc[:, :, :case["S"]] = v.transpose(1, 2)
            return {"out": _attend(case, seed, q, k, v)[0], "k_cache": kc, "v_cache": vc}
        out, _, _, _, probs, lse = _attend(case, seed, q, k, v, keep=True)
        return {"out": out, "probs": probs, "lse": lse}
