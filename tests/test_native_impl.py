"""The operator's CUDA-key implementation: the compiled one (csrc/torch_binding.cpp
built implementation-only) where it is there, else the Python one; each in a
fresh process, both over the same library."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(code):
    res = subprocess.run([sys.executable, "-c", textwrap.dedent(code)], cwd=ROOT,
                         env=dict(os.environ, PYTHONPATH=ROOT), capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, (res.stdout[-2000:], res.stderr[-3000:])
    return res.stdout


@pytest.mark.parametrize("native", [True, False])
def test_registers_with_and_without_the_compiled_implementation(native):
    out = _run(f"""
        import torch
        from custom_ops_amd import fa, ops
        if not {native}:
            fa.OPS_PATH = "/nonexistent"
        ops.ensure_loaded()
        assert (fa._ops_lib is not None) == {native}
        has = torch._C._dispatch_has_kernel_for_dispatch_key
        for key in ("CUDA", "CPU", "Meta"):
            assert has("recsys_ops::mha_fwd_with_mask", key), key
        print("ok")
    """)
    assert "ok" in out


@pytest.mark.gpu
def test_compiled_implementation_matches_the_python_one():
    out = _run("""
        import torch
        from custom_ops_amd import fa, ops
        ops.ensure_loaded()
        assert fa._ops_lib is not None
        for b, h, hk, sq, sk, d, dt in [(1, 8, 8, 100, 200, 128, torch.float16), (2, 4, 2, 300, 777, 64, torch.bfloat16),
                                        (1, 16, 16, 128, 8192, 128, torch.bfloat16), (2, 4, 4, 0, 8, 64, torch.bfloat16)]:
            q = torch.randn(b, h, sq, d, device="cuda").to(dt)
            k = torch.randn(b, hk, sk, d, device="cuda").to(dt)
            m = torch.zeros(b, 1, sq, sk, device="cuda", dtype=dt)
            side = torch.cuda.Stream()
            side.wait_stream(torch.cuda.current_stream())
            with torch.cuda.stream(side):          # the current stream, not the default one
                out = ops.mha_fwd_with_mask(q, k, k, m)
            torch.cuda.current_stream().wait_stream(side)
            assert torch.equal(out, fa.mha_fwd_with_mask_hip(q, k, k, m))
        for bad in (q.float(), q[..., :32].contiguous(), q.transpose(1, 2)):
            msgs = []
            for f in (ops.mha_fwd_with_mask, fa.mha_fwd_with_mask_hip):
                try:
                    f(bad, k, k, m)
                except RuntimeError as e:
                    msgs.append(str(e).splitlines()[0])
            assert len(msgs) == 2 and msgs[0] == msgs[1], msgs
        print("ok")
    """)
    assert "ok" in out
