"""mi355_fa_fwd_noalloc touches its per-GPU scratch array only for what a launch
needs. Without a GPU the entry point stops where it first asks for a device, and
its message says where that was: at the array, or at the launch."""
import ctypes

import pytest
import torch

from custom_ops_amd import _lib


@pytest.fixture(autouse=True)
def no_gpu():
    if torch.cuda.is_available():
        pytest.skip("pointers of this test are not memory")


def _noalloc(b, h, sq, sk, num_splits=0):
    d = 128
    p = _lib.Params(*[1 << 20] * 5, h * sq * d, sq * d, d, h * sk * d, sk * d, d, h * sk * d, sk * d, d,
                    h * sq * d, sq * d, d, sq * sk, sk, b, h, h, sq, sk, sq, sk, d, _lib.BF16, d ** -0.5, num_splits)
    lib = _lib.load()
    err = ctypes.create_string_buffer(512)
    rc = lib.mi355_fa_fwd_noalloc(ctypes.byref(p), None, err, 512)
    assert rc == _lib.EDEVICE
    return lib.mi355_fa_workspace_bytes(ctypes.byref(p)), err.value.decode()


def test_optional_words_stay_out_of_the_scratch():
    optional, msg = _noalloc(4, 16, 2048, 2048)    # the shared scan's words only
    assert optional > 0
    assert "not gfx950" in msg, msg


def test_partials_go_to_the_scratch():
    need, msg = _noalloc(1, 16, 128, 32768)
    assert need > 0
    assert "no current HIP device" in msg, msg
