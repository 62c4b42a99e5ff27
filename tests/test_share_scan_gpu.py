"""Unsplit ping-pong launches of more than one round: sampled probe, live ranges
from the scan that the head groups of a row block share, longest-first order.
Unsplit narrowing adds and leaves out exact zeros only, so every output is bit
for bit that of ``Variant(live=-1)``; replays of a captured launch (which carry
one launch tag) see the mask of their own replay."""
import pytest
import torch

from tests._ref import assert_close, ref_attn_torch

pytestmark = pytest.mark.gpu
NEG = float("-inf")

SHAPES = [  # b, h, hk, sq, sk: order 3 with 4 and 8 heads at a time, order 4, neither (no shared scan)
    (4, 16, 16, 2048, 2048), (8, 16, 16, 1000, 1024), (2, 32, 8, 2048, 1536), (3, 14, 14, 2040, 1000),
]


def _mask(kind, b, sq, sk):
    i = torch.arange(sq, device="cuda").view(-1, 1)
    j = torch.arange(sk, device="cuda").view(1, -1)
    m = torch.zeros(b, 1, sq, sk, device="cuda", dtype=torch.bfloat16)
    off = sk - sq
    if kind == "causal":
        m.masked_fill_(j > i + off, NEG)
    elif kind == "window":
        m.masked_fill_((j > i + off) | (j <= i + off - 200), NEG)
    elif kind == "one_row":      # one row of each 256 sees the last key, the others only key 70
        m.masked_fill_(torch.where(i % 256 == 131, j != sk - 1, j != 70), NEG)
    elif kind == "dead":         # no visible entry in the first batch
        m[0] = NEG
    elif kind == "stripe":
        m.masked_fill_((j < 300) | (j > 420), NEG)
    return m


def _qkv(b, h, hk, sq, sk, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [(torch.randn(b, n, s, 128, generator=g, device="cuda") * 0.5).bfloat16()
            for n, s in ((h, sq), (hk, sk), (hk, sk))]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_shared_scan_is_bit_identical(gpu, shape):
    from custom_ops_amd import Variant, mha_fwd_with_mask
    b, h, hk, sq, sk = shape
    q, k, v = _qkv(b, h, hk, sq, sk, 21)
    for kind in ("zero", "causal", "window", "one_row", "dead", "stripe"):
        m = _mask(kind, b, sq, sk)
        want = mha_fwd_with_mask(q, k, v, m, num_splits=1, variant=Variant(waves=8, live=-1))
        for var in (Variant(waves=8), Variant(waves=8, order=1), Variant(waves=8, order=2)):
            got = mha_fwd_with_mask(q, k, v, m, num_splits=1, variant=var)
            torch.cuda.synchronize()
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (kind, var)
        if kind in ("causal", "one_row"):
            assert_close(want[:1, :2], ref_attn_torch(q[:1, :2], k[:1, : max(1, 2 * hk // h)],
                                                      v[:1, : max(1, 2 * hk // h)], m[:1]), kind)


def test_shared_scan_under_graph_replay(gpu):
    from custom_ops_amd import Variant, mha_fwd_with_mask
    b, h, hk, sq, sk = SHAPES[0]
    q, k, v = _qkv(b, h, hk, sq, sk, 22)
    m = _mask("causal", b, sq, sk)
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        mha_fwd_with_mask(q, k, v, m)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        out = mha_fwd_with_mask(q, k, v, m)
    for kind in ("causal", "window", "zero", "stripe", "dead", "one_row", "causal"):
        m.copy_(_mask(kind, b, sq, sk))
        graph.replay()
        torch.cuda.synchronize()
        want = mha_fwd_with_mask(q, k, v, m, num_splits=1, variant=Variant(waves=8, live=-1))
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), want.view(torch.int16)), kind
