"""Timed cases of ``ops.mha_fwd_with_mask``: what its callers have it do, from
the smallest call to the benchmark shapes.

A case is a shape (B, H, Hk, Sq, Sk, d), a data type and a kind of additive
mask (0 = visible, -inf = blocked, other values = bias):

  zero      nothing blocked (basic attention through the same call)
  random    10 % of the entries blocked, column 0 visible (item-level masks)
  causal    keys up to the query's own position (aligned at the bottom right)
  window    the last ``Sk // 4`` keys up to the query's own position
  padding   whole keys blocked past each sequence's length (batches of unequal
            length; lengths spread evenly from Sk down to about Sk / 2)
  bias      a finite distance bias, -|distance| / 16 capped at -30, nothing blocked
  ragged    window of 1024 keys, keys of the last sequence padded, 5 % blocked

The op is forward only, so prefill (Sq ~ Sk), long-context (few queries, many
keys) and decode (Sq = 1) are its directions.
"""
from __future__ import annotations

import math

import torch

NEG_INF = float("-inf")
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _case(name, B, H, Hk, Sq, Sk, d, dtype, mask):
    c = {"B": B, "H": H, "Hk": Hk, "Sq": Sq, "Sk": Sk, "d": d, "dtype": dtype, "mask": mask}
    return dict(c, name=name) if name else c


def listed():
    return [
        # one short request: latency of a single call, nothing fills the chip
        _case("short_fp16", 1, 8, 8, 100, 200, 128, "fp16", "random"),
        # the basic example: a small batch, 64-wide heads
        _case("basic_d64", 2, 8, 8, 512, 512, 64, "bf16", "causal"),
        # the GQA example, mid-sized
        _case("gqa_mid", 2, 16, 4, 1024, 1024, 128, "bf16", "random"),
        # the benchmark shape: item-level random mask, 128-wide heads
        _case("standard", 4, 16, 16, 2048, 2048, 128, "bf16", "random"),
        # the same batch as a causal prefill, the commonest mask of all
        _case("causal", 4, 16, 16, 2048, 2048, 128, "bf16", "causal"),
        # GQA at the benchmark shape in the other data type
        _case("gqa_fp16", 4, 16, 4, 2048, 2048, 128, "fp16", "random"),
        # 64-wide heads at the benchmark shape
        _case("standard_d64", 4, 16, 16, 2048, 2048, 64, "bf16", "random"),
        # Sk not a multiple of 8 (mask rows unaligned), dense mask
        _case("ragged_dense", 4, 16, 4, 2048, 2053, 128, "bf16", "random"),
        # ragged and structured: sliding window, padding and item-level blocks
        _case("ragged_window", 2, 16, 4, 1000, 4099, 128, "bf16", "ragged"),
        # few queries over a long context, all heads: K/V streams from memory
        _case("long_context", 1, 16, 16, 128, 32768, 128, "bf16", "random"),
        # the same for a single head: a grid far too small for the chip
        _case("long_one_head", 1, 1, 1, 128, 32768, 128, "bf16", "random"),
        # decode step of a batch of unequal lengths
        _case("decode", 16, 16, 4, 1, 8192, 128, "bf16", "padding"),
    ]


#: a drawn case does no more than the largest listed one
_MAX_FLOPS = 4.0 * 4 * 16 * 2048 * 2048 * 128
_MAX_BYTES = 280e6


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    while True:
        kind = rng.choice(("prefill", "prefill", "prefill", "long", "decode"))
        ratio = rng.choice((1, 1, 2, 3, 4, 8))
        Hk = rng.choice((1, 2, 4, 8, 16))
        H = Hk * ratio
        if H > 32:
            continue
        d = rng.choice((64, 128, 128))
        dtype = rng.choice(("bf16", "bf16", "fp16"))
        if kind == "prefill":
            B = rng.choice((1, 2, 3, 4))
            Sq = _log_int(rng, 64, 2500)
            Sk = Sq if rng.random() < 0.5 else Sq + _log_int(rng, 1, 4096)
            mask = rng.choice(("zero", "random", "random", "causal", "causal", "window", "padding", "bias"))
        elif kind == "long":
            B, Sq, Sk = rng.choice((1, 1, 2)), _log_int(rng, 16, 256), _log_int(rng, 4096, 33000)
            mask = rng.choice(("zero", "random", "causal", "window"))
        else:
            B, Sq, Sk = _log_int(rng, 1, 32), 1, _log_int(rng, 100, 33000)
            mask = rng.choice(("zero", "padding", "random"))
        if rng.random() < 0.5:   # half of the sequence lengths are whole multiples of 8
            Sk = max(8, Sk // 8 * 8)
            Sq = min(Sq, Sk) if kind == "prefill" else Sq
        c = _case(None, B, H, Hk, Sq, Sk, d, dtype, mask)
        if 4.0 * B * H * Sq * Sk * d <= _MAX_FLOPS and _all_bytes(c) <= _MAX_BYTES:
            return c


def _all_bytes(c):
    rows_q, rows_k = c["B"] * c["H"] * c["Sq"], c["B"] * c["Hk"] * c["Sk"]
    return 2 * (2 * rows_q * c["d"] + 2 * rows_k * c["d"] + c["B"] * c["Sq"] * c["Sk"])


def _length(c, b):
    """Sequence b's length under a padding mask."""
    return max(1, c["Sk"] - b * (c["Sk"] // (2 * c["B"])))


def _visible(c, device):
    """The structure of the mask (without its random part): bool, broadcastable
    to [B, Sq, Sk]; None when nothing is blocked."""
    Sq, Sk, kind = c["Sq"], c["Sk"], c["mask"]
    if kind in ("zero", "random", "bias"):
        return None
    i = torch.arange(Sq, device=device).view(1, Sq, 1) + (Sk - Sq)
    j = torch.arange(Sk, device=device).view(1, 1, Sk)
    if kind == "causal":
        return j <= i
    if kind == "window":
        return (j <= i) & (j > i - max(1, Sk // 4))
    lens = torch.tensor([_length(c, b) for b in range(c["B"])], device=device).view(-1, 1, 1)
    if kind == "padding":
        return j < lens
    pad = torch.full_like(lens, Sk)
    if c["B"] > 1:
        pad[-1] = Sk - min(300, Sk // 4)
    return (j <= i) & (j > i - 1024) & (j < pad)


def _inputs(c, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    dt = DTYPES[c["dtype"]]
    B, H, Hk, Sq, Sk, d = (c[n] for n in ("B", "H", "Hk", "Sq", "Sk", "d"))

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=torch.float32).to(dt)

    q, k, v = normal(B, H, Sq, d), normal(B, Hk, Sk, d), normal(B, Hk, Sk, d)
    mask = torch.zeros(B, Sq, Sk, device=dev, dtype=dt)
    if c["mask"] == "bias":
        i = torch.arange(Sq, device=dev).view(1, Sq, 1) + (Sk - Sq)
        j = torch.arange(Sk, device=dev).view(1, 1, Sk)
        mask += (-(i - j).abs().float() / 16).clamp_min(-30.0).to(dt)
    vis = _visible(c, dev)
    if vis is not None:
        mask.masked_fill_(~vis, NEG_INF)
    share = {"random": 0.10, "ragged": 0.05}.get(c["mask"], 0.0)
    if share:
        blocked = torch.rand(B, Sq, Sk, generator=g, device=dev) < share
        if c["mask"] == "random":
            blocked[..., 0] = False
        mask.masked_fill_(blocked, NEG_INF)
    return q, k, v, mask.view(B, 1, Sq, Sk)


def prepare(case, seed):
    """Inputs on the device; the library is loaded as a program's import does."""
    from custom_ops_amd import ops

    ops.ensure_loaded()
    return (ops,) + _inputs(case, seed)


def run(state):
    ops, q, k, v, mask = state
    return ops.mha_fwd_with_mask(q, k, v, mask)


def _pairs(c):
    """(query, key) pairs per head that the structure of the mask leaves, and the keys any query sees."""
    B, Sq, Sk, kind = c["B"], c["Sq"], c["Sk"], c["mask"]
    pairs = keys = 0
    for b in range(B):
        end = Sk
        if kind == "padding":
            end = _length(c, b)
        elif kind == "ragged" and b == B - 1 and B > 1:
            end = Sk - min(300, Sk // 4)
        width = {"window": max(1, Sk // 4), "ragged": 1024}.get(kind, Sk + Sq)
        lo, hi = end, 0
        for i in range(Sq):
            last = min(end, i + (Sk - Sq) + 1) if kind in ("causal", "window", "ragged") else end
            first = max(0, i + (Sk - Sq) + 1 - width) if kind in ("window", "ragged") else 0
            if last > first:
                pairs += last - first
                lo, hi = min(lo, first), max(hi, last)
        keys += max(0, hi - lo)
    return pairs, keys


def work(case):
    """Each input read once and the output written once; two products over the pairs the mask's structure
    leaves (a randomly blocked pair still counts: no tile is free of the others). Keys no query sees need no
    reading; the mask itself has to be read."""
    c = case
    pairs, keys = _pairs(c)
    n_q = c["B"] * c["H"] * c["Sq"] * c["d"]
    n_kv = c["Hk"] * keys * c["d"]
    return {"bytes": 2.0 * (2 * n_q + 2 * n_kv + c["B"] * c["Sq"] * c["Sk"]),
            "flops": 4.0 * c["H"] * c["d"] * pairs}


def tolerance(case):
    """Rounding of P and of the output (and of split partials) to the data type."""
    return {"rel": 1e-2, "max": 0.1} if case["dtype"] == "bf16" else {"rel": 1.5e-3, "max": 0.02}


def exact(case, seed):
    q, k, v, mask = _inputs(case, seed)
    B, H, Sq, d = q.shape
    ratio = H // k.shape[1]
    out = torch.empty(B, H, Sq, d, dtype=torch.float64, device=q.device)
    for b in range(B):
        m = mask[b, 0].double()
        for h in range(H):
            kt = k[b, h // ratio].double().t().contiguous()
            s = (q[b, h].double() @ kt) / math.sqrt(d) + m
            top = s.amax(dim=-1, keepdim=True)
            p = torch.exp(s - torch.where(torch.isinf(top), torch.zeros_like(top), top))
            total = p.sum(dim=-1, keepdim=True)
            out[b, h] = (p @ v[b, h // ratio].double()) / torch.where(total == 0, torch.ones_like(total), total)
    return out
