"""64-wide heads in bf16 with a softmax scale whose reciprocal is no bf16 value
(the C ABI's ``scale_softmax``; the operator's own 1/8 has one): the 8-wave
kernel multiplies the mask by the fp32 reciprocal, bit for bit as with
``Variant(mask_mfma=-1)``, and small grids that this kernel would serve do not go
to the key streams, whose masks are weighed by bf16(1/scale)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _run(q, k, v, mask, scale, splits=1, variant=None):
    from custom_ops_amd import _lib
    from custom_ops_amd.fa import make_params
    out = torch.full_like(q, float("nan"))
    p = make_params(q, k, v, mask, out, splits, variant)
    p.scale_softmax = scale
    n = _lib.workspace_bytes(p)
    ws = torch.empty(max(n, 1), dtype=torch.uint8, device="cuda")
    p.workspace, p.workspace_bytes = ws.data_ptr(), n
    _lib.fwd(p, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    return out


def _exact(q, k, v, mask, scale):
    s = (q.double() @ k.double().transpose(-1, -2).contiguous()) * scale + mask.double()
    return torch.softmax(s, -1) @ v.double()


@pytest.mark.parametrize("sk", [640, 637])   # aligned rows, staged ones
@pytest.mark.parametrize("scale", [0.09, 0.125, 1 / 7.0])
def test_bias_is_scaled_in_fp32(gpu, scale, sk):
    from custom_ops_amd import Variant
    b, h, sq, d = 2, 4, 300, 64
    g = torch.Generator().manual_seed(3)
    q, k, v = (torch.randn(b, h, s, d, generator=g).bfloat16().cuda() for s in (sq, sk, sk))
    # a ramp down to -60: 0.13 % of it is 0.08
    i, j = torch.arange(sq).view(-1, 1), torch.arange(sk).view(1, -1)
    m = (-(i + sk - sq - j).abs().float() / 8).clamp_min(-60.0).expand(b, 1, sq, sk).bfloat16().contiguous().cuda()
    want = _run(q, k, v, m, scale, 1, Variant(waves=8, mask_mfma=-1))
    got = _run(q, k, v, m, scale, 1, Variant(waves=8))
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
    err = ((got.double() - _exact(q, k, v, m, scale)).norm() / _exact(q, k, v, m, scale).norm()).item()
    assert err < 4e-3, err


@pytest.mark.parametrize("shape", [(3, 16, 8, 662, 760), (16, 4, 4, 700, 777)], ids=lambda s: "x".join(map(str, s)))
def test_small_grids_keep_the_fp32_weight(gpu, shape):
    """Shapes whose tile plan is the 8-wave kernel, unsplit, and whose default plan
    at the operator's scale is the streams (4 per workgroup)."""
    from custom_ops_amd import Variant
    b, h, hk, sq, sk = shape
    g = torch.Generator(device="cuda").manual_seed(4)
    q, k, v = (torch.randn(b, n, s, 64, generator=g, device="cuda").bfloat16()
               for n, s in ((h, sq), (hk, sk), (hk, sk)))
    m = (torch.randn(b, 1, sq, sk, generator=g, device="cuda") * 20).bfloat16()
    pairs = ((0.09, Variant(waves=8, mask_mfma=-1)), (0.125, Variant(waves=1)))
    for scale, var in pairs:
        got, want = _run(q, k, v, m, scale, 0), _run(q, k, v, m, scale, 1, var)
        assert torch.equal(got.view(torch.int16), want.view(torch.int16)), scale
