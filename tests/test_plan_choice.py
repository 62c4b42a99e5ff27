"""Which calls the plan gives to the key streams: those where they promise to be
well below the tile plan. Calls near the line, and grids of more than one round,
keep the tile kernels (seen from the workspace: the streams need one for fp32
partials only, the tile kernels for 16-bit partials with tickets, and for the
staged copy of a mask with unaligned rows)."""
import ctypes

import pytest

TILE = [  # more than one round, near the line: measured 0.73 - 0.94 times as fast with the streams
    (2, 8, 8, 2205, 2205, 128), (3, 8, 1, 1604, 1604, 128), (3, 8, 1, 1786, 1786, 128), (2, 8, 8, 1132, 1132, 128),
    (3, 8, 2, 1469, 1658, 128), (2, 24, 8, 668, 671, 128),
]
STREAMS = [  # (and the smallest calls, decode, one long head)
    (1, 8, 8, 100, 200, 128), (2, 8, 8, 512, 512, 64), (16, 16, 4, 1, 8192, 128), (1, 1, 1, 128, 32768, 128),
    (10, 8, 4, 1, 2162, 128), (1, 6, 2, 216, 344, 64), (3, 3, 1, 254, 297, 128), (1, 16, 16, 1310, 1310, 64),
]


def _plan(b, h, hk, sq, sk, d):
    """(splits, workspace bytes, bytes of the streams' partials)"""
    from custom_ops_amd import _lib
    p = _lib.Params(q=16, k=16, v=16, mask=16, o=16, mask_batch_stride=sq * sk, mask_row_stride=sk,
                    b=b, h=h, h_k=hk, seqlen_q=sq, seqlen_k=sk, mask_seqlen_q=sq, mask_seqlen_k=sk, d=d,
                    dtype=_lib.BF16, scale_softmax=d ** -0.5)
    lib = _lib.load()
    s = lib.mi355_fa_num_splits(ctypes.byref(p))
    up = lambda n: (n + 255) // 256 * 256
    rows = s * b * h * sq
    return s, lib.mi355_fa_workspace_bytes(ctypes.byref(p)), up(rows * d * 4) + up(rows * 4) if s > 1 else 0


@pytest.mark.parametrize("shape", TILE, ids=lambda s: "x".join(map(str, s)))
def test_calls_near_the_line_keep_the_tile_kernels(shape):
    _, need, streams = _plan(*shape)
    assert need != streams and need > 0


@pytest.mark.parametrize("shape", STREAMS, ids=lambda s: "x".join(map(str, s)))
def test_small_grids_go_to_the_streams(shape):
    _, need, streams = _plan(*shape)
    assert need == streams
