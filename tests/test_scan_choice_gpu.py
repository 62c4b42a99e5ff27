"""Which unsplit ping-pong launches look for their live range together: not where
at most a few tiles are blocked at an end (keys padded by a tile or two; the words
of the shared scan stay as they were), and never past what it takes: with words,
without them, and where head groups straddle a round, every output is bit for bit
that of a launch that does not narrow."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
NEG = float("-inf")
PATTERN = 0x5A

SHAPES = [(4, 16, 16, 2048, 2048), (8, 7, 7, 2048, 2048), (8, 16, 16, 1000, 520), (4, 32, 32, 1024, 4104)]


def _mask(kind, b, sq, sk):
    i = torch.arange(sq, device="cuda").view(-1, 1)
    j = torch.arange(sk, device="cuda").view(1, -1)
    m = torch.zeros(b, 1, sq, sk, device="cuda", dtype=torch.bfloat16)
    dead = {"pad1": j >= sk - 64, "pad2": j >= sk - 130, "left1": (j < 64) & (i >= 0), "left4": j < 256,
            "both3": (j < 192) | (j >= sk - 192), "pad9": j >= sk - 9 * 64,
            "causal": j > i + (sk - sq), "anticausal": j < i, "middle": (j < sk // 2 - 40) | (j > sk // 2 + 40),
            "odd_rows": (j < 300) & (i % 2 == 0) | (j > sk - 300) & (i % 2 == 1)}[kind]
    return m.masked_fill_(dead, NEG)


def _launch(q, k, v, m, words, variant=None):
    from custom_ops_amd import _lib
    from custom_ops_amd.fa import make_params
    lib = _lib.load()
    out = torch.empty_like(q)
    p = make_params(q, k, v, m, out, 0, variant)
    n = lib.mi355_fa_workspace_bytes(ctypes.byref(p))
    assert n > 0
    ws = torch.full((n,), PATTERN, dtype=torch.uint8, device="cuda")
    if words:
        p.workspace, p.workspace_bytes = ws.data_ptr(), n
    _lib.fwd(p, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return out, ws


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_bits_with_and_without_words(gpu, shape):
    from custom_ops_amd import Variant, mha_fwd_with_mask
    b, h, hk, sq, sk = shape
    g = torch.Generator(device="cuda").manual_seed(31)
    q, k, v = [(torch.randn(b, n, s, 128, generator=g, device="cuda") * 0.5).bfloat16()
               for n, s in ((h, sq), (hk, sk), (hk, sk))]
    shared = {}
    for kind in ("pad1", "pad2", "left1", "left4", "both3", "pad9", "causal", "anticausal", "middle", "odd_rows"):
        m = _mask(kind, b, sq, sk)
        want = mha_fwd_with_mask(q, k, v, m, num_splits=1, variant=Variant(waves=8, live=-1))
        for words in (True, False):
            out, ws = _launch(q, k, v, m, words)
            assert torch.equal(out.view(torch.int16), want.view(torch.int16)), (kind, words)
            if words:
                x = ws.view(torch.int64)
                untouched = x == int.from_bytes(bytes([PATTERN]) * 8, "little")
                assert bool((untouched | (x == 0)).all()), kind     # every word published was cleared
                shared[kind] = not bool(untouched.all())
            else:
                assert bool((ws == PATTERN).all())
    for kind in ("pad1", "pad2", "left1", "left4", "both3"):
        assert not shared[kind], kind
    if sk >= 2048:
        assert shared["causal"] and shared["middle"]
