"""Mask entries past Sk are blocked whatever they hold: +inf and NaN in the pad
columns of a wider mask, in the memory behind an exact one, and in the LDS that
out-of-range DMA lanes leave as the kernel before left it. Every kernel form
gives, bit for bit, the output of the same launch over finite pads (a bf16 mask
is added on the matrix core, where a zero of the selector times such an entry
would be NaN in every key of the row)."""
import pytest
import torch

from tests._ref import assert_close, ref_attn_torch

pytestmark = pytest.mark.gpu
NEG = float("-inf")

FORMS = {   # name: (d, Variant fields, splits)
    "streams4": (128, {"waves": 1}, 1),
    "streams8": (128, {"waves": 2}, 2),
    "streams4_d64": (64, {"waves": 1}, 3),
    "streams8_d64": (64, {"waves": 2}, 1),
    "waves4": (128, {"waves": 4, "deep": -1}, 1),
    "waves4_deep": (128, {"waves": 4}, 2),
    "waves4_d64": (64, {"waves": 4}, 1),
    "waves8_d64": (64, {"waves": 8}, 1),
    "waves8_d64_split": (64, {"waves": 8}, 2),
    "compiled": (128, {"waves": 8, "loop": -1}, 1),
    "pingpong": (128, {"waves": 8, "loop": 3}, 1),
    "pingpong_split": (128, {"waves": 8, "loop": 3}, 2),
    "rows32": (128, {"waves": 8, "loop": 1}, 1),
    "rows64": (128, {"waves": 8, "loop": 2}, 2),
}
# Sk, mask columns: a tail inside a 16-byte unit; whole units; one tile or none
# before it; unaligned rows (staged for the tile kernels)
SHAPES = [(53, 56), (200, 200), (200, 264), (333, 336), (301, 301), (76, 83), (520, 520)]


def _run(q, k, v, mask, form):
    from custom_ops_amd import Variant, mha_fwd_with_mask
    _, var, splits = FORMS[form]
    return mha_fwd_with_mask(q, k, v, mask, num_splits=splits, variant=Variant(**var))


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16], ids=["bf16", "fp16"])
@pytest.mark.parametrize("form", sorted(FORMS))
def test_entries_past_sk_never_reach_a_score(gpu, form, dt):
    d = FORMS[form][0]
    b, h, hk, sq = 2, 4, 2, 67
    for sk, cols in SHAPES:
        g = torch.Generator().manual_seed(sk * 1000 + cols)
        q, k, v = ((torch.randn(b, n, s, d, generator=g) * 0.5).to(dt).cuda()
                   for n, s in ((h, sq), (hk, sk), (hk, sk)))
        vis = torch.zeros(b, 1, sq, sk).masked_fill(torch.rand(b, 1, sq, sk, generator=g) < 0.2, NEG)
        vis[..., ::7] = -0.5
        vis[:, :, 5] = NEG

        def mask(pad):
            """[b, 1, sq, cols], columns from sk on and 64 entries behind it: pad"""
            store = torch.full((b * sq * cols + 64,), pad).to(dt)
            m = store[:b * sq * cols].view(b, 1, sq, cols)
            m[..., :sk] = vis.to(dt)
            return store.cuda()[:b * sq * cols].view(b, 1, sq, cols)

        want = _run(q, k, v, mask(0.0), form)
        assert_close(want, ref_attn_torch(q, k, v, vis.to(dt).cuda()), f"{form} {sk} {cols}")
        for pad in (float("inf"), float("nan"), NEG):
            m = mask(pad)
            nan = torch.full_like(k, float("nan"))
            _run(q * float("nan"), nan, nan, torch.full_like(m, float("nan")), form)   # NaN all over the LDS
            got = _run(q, k, v, m, form)
            torch.cuda.synchronize()
            assert torch.equal(got.view(torch.int16), want.view(torch.int16)), (form, sk, cols, pad)
        if cols == sk:   # behind a row's Sk stands the next row: its NaN stays its own
            m = mask(0.0)
            m[:, :, 9, :3] = float("nan")
            m[:, :, 30, 0] = float("inf")
            got = _run(q, k, v, m, form)
            keep = torch.ones(sq, dtype=torch.bool)
            keep[[9, 30]] = False
            assert torch.equal(got[:, :, keep].view(torch.int16), want[:, :, keep].view(torch.int16)), (form, sk)
            if FORMS[form][2] == 1:   # (a split with a NaN sum counts as empty in the combine)
                assert bool(got[:, :, [9, 30]].isnan().all()), (form, sk)
