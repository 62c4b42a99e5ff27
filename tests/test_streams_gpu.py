"""The key-stream kernel (csrc/fa_streams.h: small grids, decode), forced with
``Variant(waves=1)`` (4 streams per workgroup) and ``waves=2`` (8), against the
fp32 torch restatement of the reference op at the suite's tolerance, at the
edges of its tiles: 32-key tiles, 32-row blocks of flattened (head, query)
pairs, aligned and unaligned mask rows, splits beyond the tiles there are."""
import pytest
import torch

from tests._ref import assert_close, ref_attn_torch

pytestmark = pytest.mark.gpu
NEG = float("-inf")


def _mask(kind, b, sq, sk, cols, rows, dt, g):
    i = torch.arange(sq + rows).view(-1, 1)
    j = torch.arange(sk + cols).view(1, -1)
    m = torch.zeros(b, 1, sq + rows, sk + cols)
    if kind == "causal":
        m.masked_fill_((j > i + max(0, sk - sq)).expand_as(m), NEG)
    elif kind == "top_left":          # most tiles dead
        m.masked_fill_((j > i).expand_as(m), NEG)
    elif kind == "window":
        m.masked_fill_(((j > i + sk - sq) | (j <= i + sk - sq - 40)).expand_as(m), NEG)
    elif kind == "stripes":           # dead tiles between live ones, one dead row
        m.masked_fill_(((j // 32) % 3 != 1).expand_as(m), NEG)
        m[:, :, sq // 2] = NEG
    elif kind == "bias":
        m = torch.randn(m.shape, generator=g) * 8
    elif kind == "lowest":            # the type's lowest value: finite, and overflows in bf16 after scaling
        m.masked_fill_(torch.rand(m.shape, generator=g) < 0.5, torch.finfo(dt).min)
        m[..., 0] = 0
    if kind in ("causal", "window"):
        m.masked_fill_(torch.rand(m.shape, generator=g) < 0.1, NEG)
    m[..., sk:] = 0.25                # past Sk: ignored
    m[:, :, sq:] = 0.5                # past Sq: ignored
    return m.to(dt)


CASES = [  # b, h, hk, sq, sk, d, dtype, kind, splits, extra mask columns, extra mask rows
    (1, 1, 1, 1, 1, 128, torch.bfloat16, "zero", 1, 0, 0),
    (2, 3, 1, 1, 7, 64, torch.float16, "bias", 1, 1, 0),
    (1, 8, 1, 4, 31, 128, torch.bfloat16, "zero", 1, 0, 0),      # 32 flattened rows, one tile
    (1, 4, 4, 31, 32, 64, torch.bfloat16, "causal", 1, 0, 1),
    (2, 6, 2, 11, 33, 128, torch.float16, "window", 1, 0, 0),    # 33 rows per KV head
    (1, 2, 2, 33, 129, 128, torch.bfloat16, "stripes", 1, 7, 3),
    (2, 4, 2, 100, 257, 128, torch.bfloat16, "causal", 2, 0, 0),
    (1, 4, 1, 65, 500, 64, torch.float16, "top_left", 3, 3, 0),
    (3, 2, 1, 77, 1031, 128, torch.bfloat16, "window", 1, 0, 0),
    (3, 2, 1, 77, 1031, 64, torch.bfloat16, "top_left", 5, 0, 2),
    (1, 16, 2, 1, 4099, 128, torch.float16, "stripes", 16, 0, 0),
    (1, 2, 2, 40, 300, 128, torch.bfloat16, "bias", 1, 4, 0),
    (1, 2, 1, 40, 777, 64, torch.float16, "lowest", 1, 0, 0),
    (1, 2, 1, 40, 776, 128, torch.bfloat16, "lowest", 4, 0, 0),
    (1, 1, 1, 128, 2048, 128, torch.bfloat16, "causal", 64, 0, 0),   # every stream one tile, or none
    (2, 1, 1, 5, 640, 64, torch.bfloat16, "stripes", 20, 0, 0),      # 17..: the four-wave combine
]


@pytest.mark.parametrize("waves", [1, 2])
@pytest.mark.parametrize("case", range(len(CASES)))
def test_streams_match_the_reference(gpu, case, waves):
    from custom_ops_amd import Variant, mha_fwd_with_mask
    b, h, hk, sq, sk, d, dt, kind, splits, xc, xr = CASES[case]
    g = torch.Generator().manual_seed(500 + case)
    q = (torch.randn(b, h, sq, d, generator=g) * 0.5).to(dt).cuda()
    k = (torch.randn(b, hk, sk, d, generator=g) * 0.5).to(dt).cuda()
    v = (torch.randn(b, hk, sk, d, generator=g) * 0.5).to(dt).cuda()
    m = _mask(kind, b, sq, sk, xc, xr, dt, g).cuda()
    out = mha_fwd_with_mask(q, k, v, m, num_splits=splits, variant=Variant(waves=waves))
    again = mha_fwd_with_mask(q, k, v, m, num_splits=splits, variant=Variant(waves=waves))
    torch.cuda.synchronize()
    mv = m[:, :, :sq, :sk]
    if kind == "lowest" and dt == torch.bfloat16:   # mask / scale overflows to -inf, as in the reference's kernel
        mv = mv.masked_fill(mv < -1e38, NEG)
    ref = ref_attn_torch(q, k, v, mv)
    assert_close(out, ref, f"case {CASES[case]} waves {waves}")
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))
    dead = torch.isinf(mv.float()).all(-1).unsqueeze(-1).expand(b, h, sq, d)
    assert bool((out.float().masked_select(dead) == 0).all())


@pytest.mark.parametrize("waves", [1, 2])
def test_streams_take_any_strides(gpu, waves):
    """[B, S, H, d] storage for q, k, v and o (the C ABI's strides), and a mask
    that starts off a 16-byte boundary."""
    from custom_ops_amd import _lib
    from custom_ops_amd.fa import make_params
    b, h, hk, sq, sk, d = 2, 6, 2, 21, 203, 128
    g = torch.Generator().manual_seed(9)
    q, k, v = ((torch.randn(b, s, n, d, generator=g) * 0.5).bfloat16().cuda().transpose(1, 2)
               for s, n in ((sq, h), (sk, hk), (sk, hk)))
    m = _mask("causal", b, sq, sk, 0, 0, torch.bfloat16, g)
    store = torch.zeros(m.numel() + 3, dtype=torch.bfloat16, device="cuda")
    store[3:] = m.flatten().cuda()
    mask = store[3:].view(m.shape)
    out = torch.zeros(b, sq, h, d, dtype=torch.bfloat16, device="cuda").transpose(1, 2)
    var = _lib.Variant(waves=waves)
    for splits in (1, 3):
        p = make_params(q, k, v, mask, out, splits, var)
        n = _lib.workspace_bytes(p)
        ws = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
        p.workspace, p.workspace_bytes = ws.data_ptr(), n
        out.zero_()
        _lib.fwd(p, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
        assert_close(out, ref_attn_torch(q, k, v, mask), f"splits {splits}")


def test_the_plan_takes_streams_for_small_grids(gpu):
    """The default plan's output is the forced one's, bit for bit, where the
    model puts the streams well ahead; a split count set by the caller keeps the
    tile kernels."""
    from custom_ops_amd import Variant, mha_fwd_with_mask
    g = torch.Generator().manual_seed(3)
    q = torch.randn(1, 8, 100, 128, generator=g).half().cuda()
    k = torch.randn(1, 8, 200, 128, generator=g).half().cuda()
    m = _mask("causal", 1, 100, 200, 0, 0, torch.float16, g).cuda()
    plan = mha_fwd_with_mask(q, k, k, m)
    assert torch.equal(plan, mha_fwd_with_mask(q, k, k, m, num_splits=1, variant=Variant(waves=1)))
    tile = mha_fwd_with_mask(q, k, k, m, num_splits=1)
    assert torch.equal(tile, mha_fwd_with_mask(q, k, k, m, num_splits=1, variant=Variant(waves=4)))
    assert_close(plan, tile.float(), "plan against tile kernel")
