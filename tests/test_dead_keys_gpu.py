"""Key streams skip a tile whose keys are all blocked, the first tile and the one
that reaches past Sk too: NaN in K and V there (cache rows nobody has written)
reaches no row, and what a V stage held before the last tile is gone when that
tile's missing rows meet P = 0. Bit for bit the output over zeros there."""
import pytest
import torch

from tests._ref import assert_close, ref_attn_torch

pytestmark = pytest.mark.gpu
NEG = float("-inf")

# Sk, mask columns (what stands past Sk is visible), blocked key ranges
CASES = [
    (53, 53, [(0, 32)]), (53, 56, [(32, 53)]), (200, 200, [(0, 64)]), (200, 264, [(0, 96), (192, 200)]),
    (301, 301, [(0, 64), (256, 301)]), (333, 336, [(0, 320)]), (520, 520, [(0, 256), (512, 520)]),
    (1031, 1031, [(0, 992)]),
]


def _inputs(b, h, hk, sq, sk, cols, ranges, d, dt, fill):
    g = torch.Generator().manual_seed(sk + cols)
    q, k, v = (torch.randn(b, n, s, d, generator=g) * 0.5 for n, s in ((h, sq), (hk, sk), (hk, sk)))
    m = torch.zeros(b, 1, sq, cols)
    m[:, :, :, :sk].masked_fill_(torch.rand(b, 1, sq, sk, generator=g) < 0.2, NEG)
    for lo, hi in ranges:
        k[:, :, lo:hi] = fill
        v[:, :, lo:hi] = fill
        m[:, :, :, lo:hi] = NEG
    return [x.to(dt).cuda() for x in (q, k, v, m)]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("waves,splits", [(1, 1), (1, 3), (2, 1), (2, 2)])
def test_blocked_tiles_reach_no_row(gpu, waves, splits, d, dt):
    from custom_ops_amd import Variant, mha_fwd_with_mask
    for sk, cols, ranges in CASES:
        outs = []
        for fill in (0.0, float("nan")):
            q, k, v, m = _inputs(2, 4, 2, 37, sk, cols, ranges, d, dt, fill)
            outs.append(mha_fwd_with_mask(q, k, v, m, num_splits=splits, variant=Variant(waves=waves)))
            if fill == 0.0:
                assert_close(outs[0], ref_attn_torch(q, k, v, m[..., :sk]), f"{sk} {cols}")
        torch.cuda.synchronize()
        assert torch.equal(outs[1].view(torch.int16), outs[0].view(torch.int16)), (sk, cols, ranges)


@pytest.mark.parametrize("sq", [1, 20])
def test_left_padded_cache(gpu, sq):
    """The default plan over a cache whose first rows nobody has written."""
    from custom_ops_amd import ops
    for sk in (333, 1000, 4099):
        q, k, v, m = _inputs(2, 8, 2, sq, sk, sk, [(0, 128)], 128, torch.bfloat16, float("nan"))
        out = ops.mha_fwd_with_mask(q, k, v, m)
        torch.cuda.synchronize()
        assert bool(out.isfinite().all()), sk
