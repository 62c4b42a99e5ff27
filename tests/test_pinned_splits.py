"""A split count above 1 that is the plan's own, given back by the caller, is the
same plan: the answer of mi355_fa_num_splits names the launch that the caller
gets without it. (Other counts, and 1, select among the tile kernels.)"""
import ctypes

import pytest

SHAPES = [(19, 12, 4, 1, 1808, 64), (16, 16, 4, 1, 8192, 128), (1, 1, 1, 128, 32768, 128), (4, 8, 8, 1, 4099, 128),
          (1, 16, 16, 128, 32768, 128), (2, 16, 4, 1000, 4096, 128)]


def _params(b, h, hk, sq, sk, d, splits):
    from custom_ops_amd import _lib
    p = _lib.Params(q=16, k=16, v=16, mask=16, o=16, mask_batch_stride=sq * sk, mask_row_stride=sk,
                    b=b, h=h, h_k=hk, seqlen_q=sq, seqlen_k=sk, mask_seqlen_q=sq, mask_seqlen_k=sk, d=d,
                    dtype=_lib.BF16, scale_softmax=d ** -0.5, num_splits=splits)
    for n, heads, rows in (("q", h, sq), ("k", hk, sk), ("v", hk, sk), ("o", h, sq)):
        setattr(p, f"{n}_batch_stride", heads * rows * d)
        setattr(p, f"{n}_head_stride", rows * d)
        setattr(p, f"{n}_row_stride", d)
    return p


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_the_plans_own_count_given_back(shape):
    from custom_ops_amd import _lib
    lib = _lib.load()
    auto = ctypes.byref(_params(*shape, 0))
    n = lib.mi355_fa_num_splits(auto)
    assert n > 1
    need = lib.mi355_fa_workspace_bytes(auto)
    for splits in (n, n - 1 or n + 1, n):     # (the plan of the call before is not this one's)
        pinned = ctypes.byref(_params(*shape, splits))
        assert lib.mi355_fa_num_splits(pinned) == splits
        same = lib.mi355_fa_workspace_bytes(pinned) == need
        assert same or splits != n


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES[:4], ids=lambda s: "x".join(map(str, s)))
def test_the_same_bits(gpu, shape):
    import torch
    from custom_ops_amd import mha_fwd_with_mask
    from custom_ops_amd.fa import num_splits_for
    b, h, hk, sq, sk, d = shape
    g = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn(b, n, s, d, generator=g, device="cuda").bfloat16() for n, s in ((h, sq), (hk, sk), (hk, sk)))
    m = torch.zeros(b, 1, sq, sk, device="cuda", dtype=torch.bfloat16)
    want = mha_fwd_with_mask(q, k, v, m)
    got = mha_fwd_with_mask(q, k, v, m, num_splits=num_splits_for(q, k, v, m))
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
