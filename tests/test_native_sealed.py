"""Which compiled operator implementation a process opens: in strict mode the one
that the sealed sidecar names, unchanged, or none; in development the in-tree one
if it was built from the present sources for this PyTorch, or none. Without one
the Python implementation serves. Each load in a fresh process."""
import json
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _run(code):
    env = dict(os.environ, PYTHONPATH=ROOT)
    env.pop("MI355_FA_LIB", None)
    res = subprocess.run([sys.executable, "-c", textwrap.dedent(code)], cwd=ROOT, env=env,
                         capture_output=True, text=True, timeout=300)
    assert res.returncode == 0, (res.stdout[-2000:], res.stderr[-3000:])
    return res.stdout


@pytest.fixture(scope="module")
def exported(tmp_path_factory):
    """FAOps.build with the in-tree library in place of a new compilation."""
    from custom_ops_amd import build
    from custom_ops_amd.loader import FAOps
    if not os.path.exists(build.LIB_PATH):
        build.build()
    mp = pytest.MonkeyPatch()
    mp.setattr(build, "compile_checked", lambda out, flags, verbose=False: shutil.copy2(build.LIB_PATH, out))
    try:
        return FAOps().build(tmp_path_factory.mktemp("sealed"))
    finally:
        mp.undo()


def _load(lib):
    return _run(f"""
        import torch
        from custom_ops_amd import fa
        from custom_ops_amd.loader import FAOps, CustomOpsError
        try:
            FAOps().load_precompiled({str(lib)!r})
            assert torch._C._dispatch_has_kernel_for_dispatch_key("recsys_ops::mha_fwd_with_mask", "CUDA")
            print("native", fa._ops_lib and fa._ops_lib._name)
        except CustomOpsError as e:
            print("ERR", e, fa._ops_lib)
    """)


def test_strict_mode_opens_the_sealed_implementation(exported):
    md = json.loads(open(str(exported) + ".json").read())
    ops = exported.parent / md["companion"]["file"]
    assert ops.is_file()
    assert f"native {ops}" in _load(exported)


def test_strict_mode_opens_no_other(exported, tmp_path):
    for name in (exported.name, exported.name + ".json"):
        shutil.copy2(exported.parent / name, tmp_path / name)
    assert "native None" in _load(tmp_path / exported.name)     # deployed without it
    ops = json.loads(open(str(exported) + ".json").read())["companion"]["file"]
    data = bytearray((exported.parent / ops).read_bytes())
    data[4096] ^= 0xFF
    (tmp_path / ops).write_bytes(bytes(data))
    out = _load(tmp_path / exported.name)
    assert "companion digest mismatch" in out and out.rstrip().endswith("None"), out


@pytest.mark.parametrize("change", ["sources", "torch", "unstamped"])
def test_development_load_opens_no_older_build(exported, tmp_path, change):
    from custom_ops_amd import build
    ops = exported.parent / "libmi355_fa_ops.so"
    stamp = build.ops_stamp_of(str(ops))
    assert stamp == build.ops_stamp()
    other = {"sources": stamp.replace(stamp.split()[1], "0" * 64), "torch": stamp.replace("torch 2", "torch 1"),
             "unstamped": "x" * len(stamp)}[change]
    old = tmp_path / ops.name
    old.write_bytes(ops.read_bytes().replace(stamp.encode(), other.encode()))
    out = _run(f"""
        import torch
        from custom_ops_amd import fa, ops
        fa.OPS_PATH = {str(old)!r}
        ops.ensure_loaded()
        assert torch._C._dispatch_has_kernel_for_dispatch_key("recsys_ops::mha_fwd_with_mask", "CUDA")
        print("native", fa._ops_lib)
    """)
    assert "native None" in out


def test_connect_refuses_another_abi(exported):
    out = _run(f"""
        import ctypes, torch
        from custom_ops_amd import _lib
        lib = ctypes.CDLL({str(exported.parent / "libmi355_fa_ops.so")!r})
        f = lib.mi355_ops_connect
        f.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t]
        n = ctypes.sizeof(_lib.Params)
        print("rc", f(1, 1, _lib.ABI_VERSION + 1, n), f(1, 1, _lib.ABI_VERSION, n - 8))
        print("has", torch._C._dispatch_has_kernel_for_dispatch_key("recsys_ops::mha_fwd_with_mask", "CUDA")
              if torch._C._jit_get_schemas_for_operator("recsys_ops::mha_fwd_with_mask") else False)
    """)
    assert "rc 1 1" in out and "has False" in out
