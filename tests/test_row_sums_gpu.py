"""The weights of a row sum to 1: the kernels written in HIP sum the rounded P
that the PV product uses, so a constant V comes back bit for bit (fp32 order
effects, about 1e-6, are far below half an ulp of either type)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FORMS = {   # name: (d, Variant fields, splits)
    "waves8_d64": (64, {"waves": 8}, 1),
    "waves8_d64_split": (64, {"waves": 8}, 2),
    "waves8": (128, {"waves": 8, "loop": -1}, 1),
    "waves4_d64": (64, {"waves": 4}, 1),
    "waves4": (128, {"waves": 4}, 1),
    "streams4": (128, {"waves": 1}, 1),
    "streams8_d64": (64, {"waves": 2}, 3),
}


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_constant_v_comes_back(gpu, form, dt):
    """Rows of a visible key of score 0 and, a tile later, one of score 3 to 5.4:
    the running max stays (lazy rescaling), so P of the second key is any value
    up to 2^8 and its rounding most of the row's. A sum of the unrounded P would
    be off by up to half an ulp just above a power of two, which is a whole ulp of
    an output just below one."""
    from custom_ops_amd import Variant, mha_fwd_with_mask
    d, var, splits = FORMS[form]
    g = torch.Generator().manual_seed(11)
    for sq, sk, rand in ((300, 200, False), (300, 264, False), (256, 1000, True)):
        q = torch.zeros(1, 4, sq, d) if not rand else torch.randn(1, 4, sq, d, generator=g)
        k = torch.randn(1, 4, sk, d, generator=g)
        m = torch.zeros(1, 1, sq, sk)
        if rand:
            m.masked_fill_(torch.rand(m.shape, generator=g) < 0.3, float("-inf"))
            m[..., 0] = 0
        else:
            m[:] = float("-inf")
            m[..., 0] = 0
            m[..., 100] = 3 + 2.4 * torch.arange(sq) / sq
        q, k, m = q.to(dt).cuda(), k.to(dt).cuda(), m.to(dt).cuda()
        for c in (1.0, -1.0, 4.0):
            v = torch.full_like(k, c)
            out = mha_fwd_with_mask(q, k, v, m, num_splits=splits, variant=Variant(**var))
            torch.cuda.synchronize()
            assert bool((out == c).all()), (form, sq, sk, c, (out.float() - c).abs().max().item())
