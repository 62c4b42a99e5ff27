"""Split key-stream launches hold their partials in fp32: a call that the tile
plan runs unsplit, O in fp32 throughout, is no further from 64 bits when the
streams split it; and every form of the combine (few splits in one round trip,
the one-wave and 256-thread loops, four waves for many) reads such partials."""
import math

import pytest
import torch

from tests._ref import assert_close, ref_attn_torch

pytestmark = pytest.mark.gpu


def _qkv(b, h, hk, sq, sk, d, dt, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return [torch.randn(b, n, s, d, generator=g, device="cuda").to(dt) for n, s in ((h, sq), (hk, sk), (hk, sk))]


def _error(out, q, k, v):
    r = q.shape[1] // k.shape[1]
    kk, vv = (x.double().repeat_interleave(r, 1) for x in (k, v))
    p = torch.softmax((q.double() @ kk.transpose(-1, -2).contiguous()) / math.sqrt(q.shape[-1]), -1)
    want = p @ vv
    return ((out.double() - want).norm() / want.norm()).item()


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("d", [64, 128])
def test_splitting_loses_no_precision(gpu, d, dt):
    from custom_ops_amd import mha_fwd_with_mask
    from custom_ops_amd.fa import num_splits_for
    b, h, hk, sq, sk = 19, 12, 4, 1, 1808
    split = unsplit = 0.0
    for seed in range(3):
        q, k, v = _qkv(b, h, hk, sq, sk, d, dt, seed)
        m = torch.zeros(b, 1, sq, sk, device="cuda", dtype=dt)
        assert num_splits_for(q, k, v, m) > 1
        split += _error(mha_fwd_with_mask(q, k, v, m), q, k, v)
        unsplit += _error(mha_fwd_with_mask(q, k, v, m, num_splits=1), q, k, v)
    # the same roundings of P and of the output on both sides; 16-bit partials
    # add one more of the output's size: a factor of about 1.2
    assert split <= 1.03 * unsplit, (split / 3, unsplit / 3)


@pytest.mark.parametrize("waves", [1, 2])
@pytest.mark.parametrize("splits", [2, 6, 16, 24])
@pytest.mark.parametrize("shape", [(2, 8, 4, 1100, 900, 128), (1, 3, 1, 37, 1600, 64)], ids=["many_rows", "few_rows"])
def test_combine_forms(gpu, shape, splits, waves):
    from custom_ops_amd import Variant, mha_fwd_with_mask
    b, h, hk, sq, sk, d = shape
    for dt in (torch.bfloat16, torch.float16):
        q, k, v = _qkv(b, h, hk, sq, sk, d, dt, splits)
        m = torch.zeros(b, 1, sq, sk, device="cuda", dtype=dt)
        m[:, :, 2] = float("-inf")
        m[:, :, 3, 40:] = float("-inf")   # most splits of this row are empty
        out = mha_fwd_with_mask(q, k, v, m, num_splits=splits, variant=Variant(waves=waves))
        torch.cuda.synchronize()
        assert_close(out, ref_attn_torch(q, k, v, m), f"{shape} {splits} {waves}")
        assert bool((out[:, :, 2] == 0).all())
